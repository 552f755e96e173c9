// Streaming matrix-vector product for the column counts and alignments that
// the tiled kernel (si_gemv.hip) does not take.
//
// Any whole number of blocks and any 4-byte aligned x, weights at an even
// address (the byte-by-byte kernels of si_gemv.hip take the rest, and the ops
// pinned to them).
// A workgroup of 4 waves: groups of `ks` waves split the units of a row
// among them, a wave holds 4 row slots of 16 lanes, and lane k of a slot
// takes unit k of the wave's 16-unit step for RL consecutive rows (a unit is
// 32 columns, 64 for Q4_K).  Each wave stages the 16 units' x into its own
// part of LDS with coalesced loads and needs no barrier until the slices' sums
// meet; except for the 4-bit formats, the weights and x of the next step are
// requested before the current one is multiplied.  Columns past the last whole
// unit (F16 / F32) are taken two per lane by the first slice.
//
// Bound: the decode and FP32 products of the 4-bit formats (Q4_K about 2.7
// vector instructions a weight, their units busy for 0.66 of 20000 x 5120), the
// address unit (busy 0.7) on the way to HBM for the others.  The generic kernel reads
// byte by byte, a wave a row.  Against it, weights from HBM: Q4_K 5001 x 11008
// 43.5 -> 12.1 us (2.6 TB/s), Q8_0 16000 x 5120 51 -> 18 us (4.8 TB/s), F16
// 24000 x 3500 86 -> 32 us (5.2 TB/s), F32 64 x 14000 66 -> 9 us.  With 8
// waves a workgroup the grids' last wave cost more (F16 41 us).
#include "si_gemv_units.hpp"

namespace si {
namespace {

struct __attribute__((packed, aligned(2))) u32x4_a2 {
    uint32_t x, y, z, w;
};

typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));

__device__ __forceinline__ void ld4_a2(const uint8_t* p, uint32_t* v)
{
    const u32x4_a2 a = *reinterpret_cast<const u32x4_a2*>(p);
    v[0] = a.x; v[1] = a.y; v[2] = a.z; v[3] = a.w;
}

// The unit's product with x is the block decoder's, weight by weight in FP32
// (factoring the offset out of the block, sum(q x) - 8 sum(x), cancels for an
// x with a mean: zero-mean weights, x = 1 +- 0.1, Q4_0 992 columns 7.4e-7
// instead of 1.0e-7, Q4_K 11008 columns 6.6e-7 instead of 1.2e-7).  4-bit
// values need no conversion each: masked into a 16-bit field they are fp16 (n
// times 2^-24, or 1024 + n with the exponent's bits set), which v_fma_mix_f32
// multiplies in FP32.  That takes no more time than one conversion a weight
// and the sums did (Q4_K 8000 x 1792 6.85 -> 6.25 us, 5001 x 11008 12.3 ->
// 12.1, Q4_0 16000 x 992 5.6 -> 5.5).
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
    __device__ __forceinline__ float half(int, const float4* x) const
    {
        float a0 = 0.0f, a1 = 0.0f;
#pragma unroll
        for (int k = 0; k < 8; k += 2) {
            a0 = dot4_i8(q[k], x[k], a0);
            a1 = dot4_i8(q[k + 1], x[k + 1], a1);
        }
        return half_lo(d) * (a0 + a1);
    }
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
    // d sum((n - 8) x): 1024 + n as fp16 bits, less 1032 (both exact)
    __device__ __forceinline__ float half(int, const float4* x) const
    {
        float a_lo = 0.0f, a_hi = 0.0f;
#pragma unroll
        for (int k = 0; k < 4; k++) {
            a_lo = dot4(q[k], x[k], a_lo);
            a_hi = dot4(q[k] >> 4, x[4 + k], a_hi);
        }
        return half_lo(d) * (a_lo + a_hi);
    }
    // the low nibbles of v's bytes, less 8, times x
    static __device__ __forceinline__ float dot4(uint32_t v, const float4& x, float a)
    {
        const f16x2 offset = {1032, 1032};
        const f16x2 e = __builtin_bit_cast(f16x2, (v & 0x000f000fu) | 0x64006400u) - offset;          // bytes 0, 2
        const f16x2 o = __builtin_bit_cast(f16x2, ((v >> 8) & 0x000f000fu) | 0x64006400u) - offset;   // bytes 1, 3
        a = fmaf(static_cast<float>(e.x), x.x, a);
        a = fmaf(static_cast<float>(o.x), x.y, a);
        a = fmaf(static_cast<float>(e.y), x.z, a);
        return fmaf(static_cast<float>(o.y), x.w, a);
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
    // sum(w x) with w = d1 n - m1: d1 n is exact, so the one rounding of the
    // fused form is the decoder's (its scale carries the nibble's 2^24 or 2^20)
    __device__ __forceinline__ float half(int h, const float4* x) const
    {
        const float scale = dsc[h] * (h == 0 ? 0x1p24f : 0x1p20f), m1 = -dmn[h];
        const uint32_t mask = h == 0 ? 0x000f000fu : 0x00f000f0u;
        float a0 = 0.0f, a1 = 0.0f;
#pragma unroll
        for (int k = 0; k < 8; k++) {
            const f16x2 e = __builtin_bit_cast(f16x2, qs[k] & mask);          // bytes 0, 2
            const f16x2 o = __builtin_bit_cast(f16x2, (qs[k] >> 8) & mask);   // bytes 1, 3
            a0 = fmaf(fmaf(static_cast<float>(e.x), scale, m1), x[k].x, a0);
            a1 = fmaf(fmaf(static_cast<float>(o.x), scale, m1), x[k].y, a1);
            a0 = fmaf(fmaf(static_cast<float>(e.y), scale, m1), x[k].z, a0);
            a1 = fmaf(fmaf(static_cast<float>(o.y), scale, m1), x[k].w, a1);
        }
        return a0 + a1;
    }
};

// The dense units' eight chains of four products: as short as the wave a row
// of the any-shape kernel has them at a few hundred columns (F16, 260 columns:
// 7.7e-8, with two chains of 16 9.2e-8).
__device__ __forceinline__ float sum8(const float (&a)[8])
{
    return ((a[0] + a[4]) + (a[1] + a[5])) + ((a[2] + a[6]) + (a[3] + a[7]));
}

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
    __device__ __forceinline__ float half(int, const float4* x) const
    {
        float a[8] = {};
#pragma unroll
        for (int k = 0; k < 8; k++) {
            const int c = 4 * (k & 1);
            a[c] = fmaf(half_lo(v[2 * k]), x[k].x, a[c]);
            a[c + 1] = fmaf(half_hi(v[2 * k]), x[k].y, a[c + 1]);
            a[c + 2] = fmaf(half_lo(v[2 * k + 1]), x[k].z, a[c + 2]);
            a[c + 3] = fmaf(half_hi(v[2 * k + 1]), x[k].w, a[c + 3]);
        }
        return sum8(a);
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
    __device__ __forceinline__ float half(int, const float4* x) const
    {
        float a[8] = {};
#pragma unroll
        for (int k = 0; k < 8; k++) {
            const int c = 4 * (k & 1);
            a[c] = fmaf(__uint_as_float(v[4 * k]), x[k].x, a[c]);
            a[c + 1] = fmaf(__uint_as_float(v[4 * k + 1]), x[k].y, a[c + 1]);
            a[c + 2] = fmaf(__uint_as_float(v[4 * k + 2]), x[k].z, a[c + 2]);
            a[c + 3] = fmaf(__uint_as_float(v[4 * k + 3]), x[k].w, a[c + 3]);
        }
        return sum8(a);
    }
};

constexpr int STREAM_WAVES = 4;

template <int FMT, int RL, int NS>
__global__ __launch_bounds__(64 * STREAM_WAVES) void gemv_stream_kernel(Segs<NS> segs, int ks)
{
    using U = SUnit<FMT>;
    constexpr int HALVES = U::COLS / 32;              // 32-column blocks per unit
    constexpr int XPT = U::COLS / 16;                 // float4 values of x per lane and step
    constexpr bool DENSE = block_elems(FMT) == 1;
    // the 4-bit formats decode long enough for the other waves to cover a
    // step's round trip, and the registers of a second step cost waves (Q4_K
    // 20000 x 5120: 24.9 us ahead, 17.9 without; Q4_0 8000 x 5120: 9.9 and
    // 10.2; F16 24000 x 3500: 32.3 ahead, 33.7 without)
    constexpr bool AHEAD = FMT != FMT_Q4_0 && FMT != FMT_Q4_K;
    constexpr int XU = 8 * HALVES + 1;                 // float4 values of a unit in LDS, odd: 16 lanes hit distinct banks
    __shared__ float4 xs[STREAM_WAVES][16 * XU];
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
#pragma unroll
                for (int t = 0; t < RL; t++) {
                    const float v = wd[t].half(h, xv);
                    acc[t] += in ? v : 0.0f;
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
// one, 10.2 with two; 100 x 12000 4.6 and 6.3 the other way).  The 4-bit formats'
// longer decode is shared worse by two or three waves a SIMD, so theirs lies at
// three (Q4_0) and four (Q4_K): 5001 x 11008, 626 workgroups of two rows, two calls
// of Q4_K 17.8 us with one row and 20.5 with two, Q4_0 19.5 and 20.7; Q4_K 20000 x
// 5120, 2500, 18.0 and 17.5; Q4_0 16000 x 992, 1000, 5.8 and 5.5.  Four rows
// measured no faster, and F16 / F32 rows stream best alone (F16 5001 x 11007 22
// us, 27 with two).
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
        if (rows / (STREAM_WAVES / ks * 8) >= (FMT == FMT_Q8_0 ? 512 : FMT == FMT_Q4_0 ? 768 : 1024))
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
