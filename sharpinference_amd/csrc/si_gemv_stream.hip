// Streaming matrix-vector product for the column counts and alignments that
// the tiled kernel (si_gemv.hip) does not take.
//
// Any whole number of blocks and any 4-byte aligned x, weights at an even
// address (the kernel above takes the rest, and the ops pinned to it).
// A workgroup of 4 waves: groups of `ks` waves split the units of a row
// among them, a wave holds 4 row slots of 16 lanes, and lane k of a slot
// takes unit k of the wave's 16-unit step for RL consecutive rows (a unit is
// 32 columns, 64 for Q4_K).  Each wave stages the 16 units' x into its own
// part of LDS with coalesced loads and needs no barrier until the slices' sums meet; the
// weights and x of the next step are requested before the current one is
// multiplied.  Columns past the last whole unit (F16 / F32) are taken two
// per lane by the first slice.
//
// Bound: the FP32 products of the 4-bit formats (about 230 vector
// instructions per 64 weights), HBM for the others.  The generic kernel reads
// byte by byte, a wave a row.  Against it, weights from HBM: Q4_K 5001 x 11008
// 43.5 -> 11.2 us (2.8 TB/s), Q8_0 16000 x 5120 51 -> 18 us (4.8 TB/s), F16
// 24000 x 3500 86 -> 32 us (5.2 TB/s), F32 64 x 14000 66 -> 9 us.  With 8
// waves a workgroup the grids' last wave cost more (Q4_K 17 us, F16 41 us).
#include "si_gemv_units.hpp"

namespace si {
namespace {

struct __attribute__((packed, aligned(2))) u32x4_a2 {
    uint32_t x, y, z, w;
};
typedef uint32_t u32_a2 __attribute__((aligned(2)));

__device__ __forceinline__ void ld4_a2(const uint8_t* p, uint32_t* v)
{
    const u32x4_a2 a = *reinterpret_cast<const u32x4_a2*>(p);
    v[0] = a.x; v[1] = a.y; v[2] = a.z; v[3] = a.w;
}

template <int FMT>
struct SUnit;

template <>
struct SUnit<FMT_Q8_0> {
    static constexpr int COLS = 32, BYTES = 34;
    uint32_t d, q[8];
    __device__ __forceinline__ void load(const uint8_t* row, int u)
    {
        const uint8_t* p = row + static_cast<int64_t>(u) * BYTES;
        d = *reinterpret_cast<const uint16_t*>(p);
        ld4_a2(p + 2, q);
        ld4_a2(p + 18, q + 4);
    }
    __device__ __forceinline__ void prepare() {}
    __device__ __forceinline__ float half(int, const float4* x, float) const
    {
        float a0 = 0.0f, a1 = 0.0f;
#pragma unroll
        for (int k = 0; k < 8; k += 2) {
            a0 = dot4_i8(q[k], x[k], a0);
            a1 = dot4_i8(q[k + 1], x[k + 1], a1);
        }
        return half_lo(d) * (a0 + a1);
    }
    __device__ float half_exact(int h, const float4* x) const { return half(h, x, 0.0f); }
};

template <>
struct SUnit<FMT_Q4_0> {
    static constexpr int COLS = 32, BYTES = 18;
    uint32_t d, q[4];
    __device__ __forceinline__ void load(const uint8_t* row, int u)
    {
        const uint8_t* p = row + static_cast<int64_t>(u) * BYTES;
        d = *reinterpret_cast<const uint16_t*>(p);
        ld4_a2(p + 2, q);
    }
    __device__ __forceinline__ void prepare() {}
    __device__ __forceinline__ float half(int, const float4* x, float sx) const
    {
        float a_lo = 0.0f, a_hi = 0.0f;
#pragma unroll
        for (int k = 0; k < 4; k++) {
            a_lo = dot4_u8(opaque(q[k] & 0x0f0f0f0fu), x[k], a_lo);
            a_hi = dot4_u8(opaque(q[k] & 0xf0f0f0f0u), x[4 + k], a_hi);
        }
        return half_lo(d) * fmaf(-8.0f, sx, fmaf(a_hi, 0.0625f, a_lo));
    }
    // as QUnit<FMT_Q4_0>::half_exact
    __device__ float half_exact(int, const float4* x) const
    {
        float a = 0.0f;
        for (int k = 0; k < 4; k++) {
            const uint32_t t = q[k] ^ 0x88888888u;
            a = dot4_i8((t << 4) & 0xf0f0f0f0u, x[k], a);
            a = dot4_i8(t & 0xf0f0f0f0u, x[4 + k], a);
        }
        return (half_lo(d) * 0.0625f) * a;
    }
};

template <>
struct SUnit<FMT_Q4_K> : QUnit<FMT_Q4_K> {
    static constexpr int COLS = 64;
    __device__ __forceinline__ void load(const uint8_t* row, int u)
    {
        chunk = u & 3;
        const uint8_t* p = row + static_cast<int64_t>(u >> 2) * 144;
        ld4_a2(p, hd);
        ld4_a2(p + 16 + 32 * chunk, qs);
        ld4_a2(p + 32 + 32 * chunk, qs + 4);
    }
};

template <>
struct SUnit<FMT_F16> {
    static constexpr int COLS = 32, BYTES = 64;
    uint32_t v[16];
    __device__ __forceinline__ void load(const uint8_t* row, int u)
    {
        const uint8_t* p = row + static_cast<int64_t>(u) * BYTES;
#pragma unroll
        for (int i = 0; i < 4; i++)
            ld4_a2(p + 16 * i, v + 4 * i);
    }
    __device__ __forceinline__ void prepare() {}
    __device__ __forceinline__ float half(int, const float4* x, float) const
    {
        float a0 = 0.0f, a1 = 0.0f;
#pragma unroll
        for (int k = 0; k < 8; k++) {
            a0 = fmaf(half_lo(v[2 * k]), x[k].x, a0);
            a1 = fmaf(half_hi(v[2 * k]), x[k].y, a1);
            a0 = fmaf(half_lo(v[2 * k + 1]), x[k].z, a0);
            a1 = fmaf(half_hi(v[2 * k + 1]), x[k].w, a1);
        }
        return a0 + a1;
    }
};

template <>
struct SUnit<FMT_F32> {
    static constexpr int COLS = 32, BYTES = 128;
    uint32_t v[32];
    __device__ __forceinline__ void load(const uint8_t* row, int u)
    {
        const uint8_t* p = row + static_cast<int64_t>(u) * BYTES;
#pragma unroll
        for (int i = 0; i < 8; i++)
            ld4_a2(p + 16 * i, v + 4 * i);
    }
    __device__ __forceinline__ void prepare() {}
    __device__ __forceinline__ float half(int, const float4* x, float) const
    {
        float a0 = 0.0f, a1 = 0.0f;
#pragma unroll
        for (int k = 0; k < 8; k++) {
            a0 = fmaf(__uint_as_float(v[4 * k]), x[k].x, a0);
            a1 = fmaf(__uint_as_float(v[4 * k + 1]), x[k].y, a1);
            a0 = fmaf(__uint_as_float(v[4 * k + 2]), x[k].z, a0);
            a1 = fmaf(__uint_as_float(v[4 * k + 3]), x[k].w, a1);
        }
        return a0 + a1;
    }
};

constexpr int STREAM_WAVES = 4;

template <int FMT, int RL, int NS>
__global__ __launch_bounds__(64 * STREAM_WAVES) void gemv_stream_kernel(Segs<NS> segs, int ks)
{
    using U = SUnit<FMT>;
    constexpr int HALVES = U::COLS / 32;              // 32-column blocks per unit
    constexpr int XPT = U::COLS / 16;                 // float4 values of x per lane and step
    constexpr bool SUMS = FMT == FMT_Q4_0 || FMT == FMT_Q4_K;
    constexpr bool DENSE = block_elems(FMT) == 1;
    // the 4-bit formats decode long enough for the other waves to cover a
    // step's round trip, and the registers of a second step would halve
    // their number (Q4_K 5001 x 11008: 14.8 us ahead, 11.2 without; F16
    // 24000 x 3500: 32.3 ahead, 33.7 without)
    constexpr bool AHEAD = !SUMS;
    constexpr int XU = 8 * HALVES + 1;                 // float4 values of a unit in LDS, odd: 16 lanes hit distinct banks
    __shared__ float4 xs[STREAM_WAVES][16 * XU];
    __shared__ float bs[STREAM_WAVES][SUMS ? 16 * HALVES : 1];
    __shared__ float part[2][STREAM_WAVES * 4 * RL];

    const Seg& sg = segs.s[NS == 1 ? 0 : blockIdx.y];   // the op of this grid row
    const int b = static_cast<int>(blockIdx.x);
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int slice = wave & (ks - 1);                  // ks is a power of two
    const int group_rows = 4 * RL;
    const int wg_rows = STREAM_WAVES / ks * group_rows;
    const int rows = sg.rows;
    const int rb = b * wg_rows;
    if (rb >= rows)
        return;                                         // past this op's rows: the whole workgroup
    side_copy(sg, b, 64 * STREAM_WAVES);
    const int lk = lane & 15;
    const int local_row0 = wave / ks * group_rows + (lane >> 4) * RL;
    const int K = sg.blocks * block_elems(FMT);
    const int units = K / U::COLS;
    const int64_t row_bytes = static_cast<int64_t>(sg.blocks) * block_bytes(FMT);
    const bool swiglu = sg.out == OUT_SWIGLU_ROWS;

    for (int pass = 0; pass < (swiglu ? 2 : 1); pass++) {   // gate rows, then up rows
        const uint8_t* rp[RL];
#pragma unroll
        for (int t = 0; t < RL; t++)   // rows past the end repeat the last; their results are dropped
            rp[t] = sg.w + (static_cast<int64_t>(min(rb + local_row0 + t, rows - 1)) + static_cast<int64_t>(pass) * rows) *
                               row_bytes;
        float acc[RL];
#pragma unroll
        for (int t = 0; t < RL; t++)
            acc[t] = 0.0f;
        const int ntail = DENSE ? K - units * U::COLS : 0;   // columns past the last whole unit

        U w[1 + AHEAD][RL];
        float4 xr[1 + AHEAD][XPT];
        auto load = [&](int ubase, U (&wd)[RL], float4 (&xd)[XPT]) {
#pragma unroll
            for (int j = 0; j < XPT; j++) {
                const int col = min(ubase * U::COLS + 4 * (lane + 64 * j), units * U::COLS - 4);
                const u32x4 v = *reinterpret_cast<const u32x4*>(sg.x + col);   // 4-byte aligned
                xd[j] = make_float4(__uint_as_float(v.x), __uint_as_float(v.y), __uint_as_float(v.z),
                                    __uint_as_float(v.w));
            }
            const int u = min(ubase + lk, units - 1);
#pragma unroll
            for (int t = 0; t < RL; t++)
                wd[t].load(rp[t], u);
        };
        auto multiply = [&](int ubase, U (&wd)[RL], const float4 (&xd)[XPT]) {
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");   // the previous step's reads of xs come first
            __builtin_amdgcn_wave_barrier();
#pragma unroll
            for (int j = 0; j < XPT; j++) {
                const int q = lane + 64 * j;
                xs[wave][q / (8 * HALVES) * XU + q % (8 * HALVES)] = xd[j];
                if constexpr (SUMS) {
                    // a block with a non-finite or huge value stores NaN: the per-weight form
                    const bool wide = !(fabsf(xd[j].x) <= 0x1p100f && fabsf(xd[j].y) <= 0x1p100f &&
                                        fabsf(xd[j].z) <= 0x1p100f && fabsf(xd[j].w) <= 0x1p100f);
                    const float sum =
                        group_sum<8>(wide ? __builtin_nanf("") : (xd[j].x + xd[j].y) + (xd[j].z + xd[j].w));
                    if ((lane & 7) == 0)
                        bs[wave][q >> 3] = sum;
                }
            }
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
            __builtin_amdgcn_wave_barrier();
            const bool in = ubase + lk < units;
#pragma unroll
            for (int t = 0; t < RL; t++)
                wd[t].prepare();
#pragma unroll
            for (int h = 0; h < HALVES; h++) {
                float4 xv[8];
#pragma unroll
                for (int k = 0; k < 8; k++)
                    xv[k] = xs[wave][lk * XU + 8 * h + k];
                if constexpr (SUMS) {
                    const float sx = bs[wave][lk * HALVES + h];
                    if (__builtin_expect(sx == sx, 1)) {
#pragma unroll
                        for (int t = 0; t < RL; t++) {
                            const float v = wd[t].half(h, xv, sx);
                            acc[t] += in ? v : 0.0f;
                        }
                    } else if (in) {
                        for (int t = 0; t < RL; t++)
                            acc[t] += wd[t].half_exact(h, xv);
                    }
                } else {
#pragma unroll
                    for (int t = 0; t < RL; t++) {
                        const float v = wd[t].half(h, xv, 0.0f);
                        acc[t] += in ? v : 0.0f;
                    }
                }
            }
        };
        if (DENSE && ntail > 0 && slice == 0) {
            float xt[2], wt[2][RL];
#pragma unroll
            for (int i = 0; i < 2; i++) {
                const int c = min(units * U::COLS + lk + 16 * i, K - 1);
                xt[i] = sg.x[c];
#pragma unroll
                for (int t = 0; t < RL; t++)
                    wt[i][t] = elem<FMT>(rp[t] + static_cast<int64_t>(c) * block_bytes(FMT));
            }
#pragma unroll
            for (int i = 0; i < 2; i++)
#pragma unroll
                for (int t = 0; t < RL; t++)
                    acc[t] = lk + 16 * i < ntail ? fmaf(wt[i][t], xt[i], acc[t]) : acc[t];
        }
        const int stride = 16 * ks;
        int ub = 16 * slice;
        if constexpr (AHEAD) {
            if (ub < units)
                load(ub, w[0], xr[0]);
            while (ub < units) {
                if (ub + stride < units)
                    load(ub + stride, w[1], xr[1]);
                multiply(ub, w[0], xr[0]);
                ub += stride;
                if (ub >= units)
                    break;
                if (ub + stride < units)
                    load(ub + stride, w[0], xr[0]);
                multiply(ub, w[1], xr[1]);
                ub += stride;
            }
        } else {
            for (; ub < units; ub += stride) {
                load(ub, w[0], xr[0]);
                multiply(ub, w[0], xr[0]);
            }
        }
#pragma unroll
        for (int t = 0; t < RL; t++) {
            const float v = group_sum<16>(acc[t]);
            if (lk == 0)
                part[pass][(local_row0 + t) * ks + slice] = v;
        }
    }
    __syncthreads();
    const int t = threadIdx.x, r = rb + t;
    if (t >= wg_rows || r >= rows)
        return;
    float v = 0.0f, u = 0.0f;
    for (int k = 0; k < ks; k++) {   // fixed order
        v += part[0][t * ks + k];
        if (swiglu)
            u += part[1][t * ks + k];
    }
    sg.y[r] = swiglu ? silu_mul(v, u) : finish(sg, v, sg.residual ? sg.residual[r] : 0.0f, sg.residual != nullptr);
}

// Waves per row (ks): as many as give each lane at most one unit, up to 4.
// Rows per lane (RL): two rows of the block formats per staged x value where
// the grid still gives each CU two workgroups (Q8_0 24000 x 1056 13.4 us with
// one, 10.2 with two; 100 x 12000 4.6 and 6.3 the other way); four measured
// no faster, and F16 / F32 rows stream best alone (F16 5001 x 11007 22 us, 27
// with two).
template <int FMT, int RL>
hipError_t launch_stream_rows(const GemvOp* ops, int n, int ks, hipStream_t s)
{
    auto per = [ks](const GemvOp&) { return STREAM_WAVES / ks * 4 * RL; };
    if (n == 1) {
        Segs<1> t;
        const dim3 grid = fill_segs(t, ops, n, per);
        hipLaunchKernelGGL((gemv_stream_kernel<FMT, RL, 1>), grid, dim3(64 * STREAM_WAVES), 0, s, t, ks);
    } else {
        Segs<MAX_SEGS> t;
        const dim3 grid = fill_segs(t, ops, n, per);
        hipLaunchKernelGGL((gemv_stream_kernel<FMT, RL, MAX_SEGS>), grid, dim3(64 * STREAM_WAVES), 0, s, t, ks);
    }
    return hipGetLastError();
}

template <int FMT>
hipError_t launch_stream(const GemvOp* ops, int n, hipStream_t s)
{
    int64_t rows = 0, units = 1;
    for (int i = 0; i < n; i++) {
        rows += ops[i].rows;
        units = std::max(units, ops[i].cols / SUnit<FMT>::COLS);
    }
    int ks = 1;
    while (ks < STREAM_WAVES && 16 * ks < units)
        ks *= 2;
    if constexpr (is_block_quant(FMT)) {
        if (rows / (STREAM_WAVES / ks * 8) >= 512)
            return launch_stream_rows<FMT, 2>(ops, n, ks, s);
    }
    return launch_stream_rows<FMT, 1>(ops, n, ks, s);
}

}  // namespace

hipError_t launch_gemv_stream(const GemvOp* ops, int n, hipStream_t s)
{
    switch (ops[0].fmt) {
    case FMT_Q8_0: return launch_stream<FMT_Q8_0>(ops, n, s);
    case FMT_Q4_0: return launch_stream<FMT_Q4_0>(ops, n, s);
    case FMT_Q4_K: return launch_stream<FMT_Q4_K>(ops, n, s);
    case FMT_F16: return launch_stream<FMT_F16>(ops, n, s);
    case FMT_F32: return launch_stream<FMT_F32>(ops, n, s);
    default: return hipErrorInvalidValue;
    }
}

}  // namespace si
