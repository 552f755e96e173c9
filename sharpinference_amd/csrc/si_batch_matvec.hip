// The batched prefill's mat-vec y[t][o] = sum_k x[t][k] W[o][k] of up to 16
// live FP32 rows x (GpuBatchTransformerInstructions.cs:224-279), for F16
// and F32 weights with columns % 64 == 0.
//
// A workgroup of 8 waves owns 16 * WN rows of W; the waves split the
// 64-column steps of K (a contiguous run each), two steps in flight, and add
// their 16 x 16 tiles through LDS at the end in wave order: no barrier in the
// loop, and results are reproducible.  Lanes load whole lines (lane l: row l / 4,
// part l % 4 of the step) and exchange through the wave's own LDS into the
// matrix cores' order, lane (r, g) = (l % 16, l / 16): part g of row r.
//
// Products are FP32 (v_mfma_f32_16x16x4_f32), two chains a tile.
//
// Bound: HBM (F16 16384 x 3072 100 MB, F32 201 MB) with the exchange's chain
// per step.  Loaded straight into fragment order, a load instruction met 16
// rows (si_batch.hip's kernel): F16 at 16 rows, weights from HBM, 5120 x 3072
// 20.2 -> 14.2 us, 3072 x 3072 11.0 -> 7.8, 16384 x 3072 38.1 -> 25.5 (3.9
// TB/s), 3072 x 8192 27.6 -> 18.9; F32 27.7 -> 20.6, 16.2 -> 12.3, 52.1 ->
// 45.0 (4.5 TB/s), 34.4 -> 31.6.  The block formats keep the LDS ring: here they
// took 8.6 to 9.5 us for 3072 x 3072 against 8.0 to 8.6.
#include "si_batch.hpp"
#include "si_prefill_units.hpp"

namespace si {
namespace {

constexpr int MV_WAVES = 8;

// Part q (0..3) of a row's 64-column step: columns 8q .. 8q + 7 of both
// 32-column blocks, 4 (F16) or 8 (F32) words of each.
template <int FMT>
constexpr int part_words() { return FMT == FMT_F16 ? 8 : 16; }
template <int FMT>
struct Part {
    uint32_t w[part_words<FMT>()];
};

// base: the workgroup's first row plus the step (uniform); off: the lane's
// part of its row.
template <int FMT>
__device__ __forceinline__ Part<FMT> load_part(const uint8_t* base, uint32_t off)
{
    Part<FMT> r;
    off = opaque(off);
    constexpr int N = FMT == FMT_F16 ? 1 : 2;   // 16-byte loads per block
#pragma unroll
    for (int b = 0; b < 2; b++)
#pragma unroll
        for (int i = 0; i < N; i++) {
            const u32x4 v = *reinterpret_cast<const u32x4*>(base + off + 64 * N * b + 16 * i);
#pragma unroll
            for (int k = 0; k < 4; k++)
                r.w[4 * (N * b + i) + k] = v[k];
        }
    return r;
}

// The 8 weights of block b.
template <int FMT>
__device__ __forceinline__ f32x8 part_weights(const Part<FMT>& p, int b)
{
    f32x8 v;
#pragma unroll
    for (int i = 0; i < 8; i++) {
        if constexpr (FMT == FMT_F16)
            v[i] = half_bits(p.w[4 * b + i / 2] >> (16 * (i & 1)));
        else
            v[i] = __uint_as_float(p.w[8 * b + i]);
    }
    return v;
}

template <int FMT, int WN>
__global__ __launch_bounds__(64 * MV_WAVES) void batch_matvec_exchange_kernel(
    const uint8_t* __restrict__ W, const float* __restrict__ X, float* __restrict__ Y, int batch, int rows, int cols,
    int64_t row_bytes, const int32_t* __restrict__ control)
{
    constexpr int D = 2;                                  // steps in flight
    constexpr int QW = part_words<FMT>() / 4;             // 16-byte groups of a part
    constexpr int XG = 4;                                 // and of x: 1 KB each a wave
    constexpr int WAVE_WORDS = 256 * (XG + QW * WN);
    constexpr int RED_WORDS = MV_WAVES * WN * 256;
    constexpr int POOL = MV_WAVES * WAVE_WORDS > RED_WORDS ? MV_WAVES * WAVE_WORDS : RED_WORDS;
    __shared__ __attribute__((aligned(16))) uint32_t pool[POOL];
    const int n0 = static_cast<int>(blockIdx.x) * 16 * WN, t0 = static_cast<int>(blockIdx.y) * 16;
    const int live = min(control[1], batch) - t0;         // live batch rows of this tile
    if (live <= 0)
        return;                                           // the whole workgroup, before any barrier
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int steps = cols / 64;
    const int per = (steps + MV_WAVES - 1) / MV_WAVES;
    const int s0 = wave * per, mine = min(per, steps - s0);   // this wave's steps (may be none)

    const int lr = lane >> 2, lq = lane & 3;              // what the lane loads
    const int fr = lane & 15, fg = lane >> 4;             // what it multiplies
    const int wslot = 4 * lr + (lq ^ ((lr >> 2) & 3)), rslot = 4 * fr + (fg ^ ((fr >> 2) & 3));
    u32x4* const g4 = reinterpret_cast<u32x4*>(pool + wave * WAVE_WORDS);

    const uint8_t* const wb = W + static_cast<int64_t>(n0) * row_bytes;
    const uint8_t* const xb = reinterpret_cast<const uint8_t*>(X + static_cast<int64_t>(t0) * cols);
    uint32_t woff[WN];
#pragma unroll
    for (int j = 0; j < WN; j++)   // rows past the end repeat the last; their results are dropped
        woff[j] = static_cast<uint32_t>(min(16 * j + lr, rows - 1 - n0)) * static_cast<uint32_t>(row_bytes) +
                  (FMT == FMT_F16 ? 16 : 32) * lq;
    // rows past the live ones repeat the last live one
    const uint32_t xoff = static_cast<uint32_t>(min(lr, live - 1)) * static_cast<uint32_t>(4 * cols) + 32 * lq;

    f32x4 acc[WN][2];                                     // two chains of products
#pragma unroll
    for (int j = 0; j < WN; j++)
        acc[j][0] = acc[j][1] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};

    Part<FMT> raw[D][WN];
    f32x4 xr[D][4];   // block b: the part's values 0..3 and 4..7
    auto load_step = [&](int k, Part<FMT> (&wd)[WN], f32x4 (&xd)[4]) {
        const int st = s0 + k;
        const uint8_t* base = wb + static_cast<int64_t>(st) * (FMT == FMT_F16 ? 128 : 256);
        const uint8_t* xbase = xb + static_cast<int64_t>(st) * 256;
        const uint32_t o = opaque(xoff);
#pragma unroll
        for (int i = 0; i < 4; i++)
            xd[i] = *reinterpret_cast<const f32x4*>(xbase + o + 128 * (i >> 1) + 16 * (i & 1));
#pragma unroll
        for (int j = 0; j < WN; j++)
            wd[j] = load_part<FMT>(base, woff[j]);
    };
    // the step into the wave's part of LDS (a wave's LDS accesses execute in
    // order: the fences only keep the compiler's order)
    auto stage = [&](const Part<FMT> (&wd)[WN], const f32x4 (&xd)[4]) {
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
#pragma unroll
        for (int i = 0; i < 4; i++)
            g4[64 * i + wslot] = __builtin_bit_cast(u32x4, xd[i]);
#pragma unroll
        for (int j = 0; j < WN; j++)
#pragma unroll
            for (int q = 0; q < QW; q++)
                g4[64 * (XG + QW * j + q) + wslot] =
                    u32x4{wd[j].w[4 * q], wd[j].w[4 * q + 1], wd[j].w[4 * q + 2], wd[j].w[4 * q + 3]};
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
    };
    // a step staged in LDS: the next one takes its place there and the one
    // `more` (< 0: none) is requested into the registers that frees
    auto run_step = [&](Part<FMT> (&wn)[WN], f32x4 (&xn)[4], bool next, int more) {
        Part<FMT> wf[WN];
        f32x4 xf[4];
#pragma unroll
        for (int j = 0; j < WN; j++)
#pragma unroll
            for (int q = 0; q < QW; q++) {
                const u32x4 v = g4[64 * (XG + QW * j + q) + rslot];
#pragma unroll
                for (int k = 0; k < 4; k++)
                    wf[j].w[4 * q + k] = v[k];
            }
#pragma unroll
        for (int k = 0; k < 4; k++)
            xf[k] = __builtin_bit_cast(f32x4, g4[64 * k + rslot]);
        if (next)
            stage(wn, xn);
        if (more >= 0)
            load_step(more, wn, xn);
#pragma unroll
        for (int b = 0; b < 2; b++)
#pragma unroll
            for (int j = 0; j < WN; j++) {
                const f32x8 w = part_weights<FMT>(wf[j], b);
#pragma unroll
                for (int e = 0; e < 8; e++)
                    acc[j][e & 1] = __builtin_amdgcn_mfma_f32_16x16x4f32(xf[2 * b + e / 4][e & 3], w[e], acc[j][e & 1], 0, 0, 0);
            }
    };

    if (mine > 0) {
#pragma unroll
        for (int u = 0; u < D; u++)
            load_step(min(u, mine - 1), raw[u], xr[u]);
        stage(raw[0], xr[0]);
        if (D < mine)
            load_step(D, raw[0], xr[0]);
        int i = 0;
        for (; i + 2 * D < mine; i += D) {
#pragma unroll
            for (int u = 0; u < D; u++)
                run_step(raw[(u + 1) % D], xr[(u + 1) % D], true, i + u + 1 + D);
        }
#pragma unroll
        for (int u = 0; u < 2 * D; u++)
            if (i + u < mine)
                run_step(raw[(u + 1) % D], xr[(u + 1) % D], i + u + 1 < mine, i + u + 1 + D < mine ? i + u + 1 + D : -1);
    }

    // the waves' tiles meet in LDS; tile j is summed in wave order and stored
    // by wave j
    __syncthreads();
    f32x4* red = reinterpret_cast<f32x4*>(pool);
#pragma unroll
    for (int j = 0; j < WN; j++)
        red[(wave * WN + j) * 64 + lane] = acc[j][0] + acc[j][1];
    __syncthreads();
    if (wave < WN) {
        f32x4 v = red[wave * 64 + lane];
#pragma unroll
        for (int w = 1; w < MV_WAVES; w++)
            v += red[(w * WN + wave) * 64 + lane];
        const int o = n0 + 16 * wave + fr;
#pragma unroll
        for (int e = 0; e < 4; e++) {
            const int i = 4 * fg + e;
            if (i < live && o < rows)
                Y[static_cast<int64_t>(t0 + i) * rows + o] = v[e];
        }
    }
}

template <int FMT, int WN>
void launch_tile(const uint8_t* w, const float* x, float* y, int batch, int64_t rows, int64_t cols,
                 const int32_t* control, hipStream_t s)
{
    const dim3 grid(static_cast<unsigned>((rows + 16 * WN - 1) / (16 * WN)), static_cast<unsigned>((batch + 15) / 16));
    hipLaunchKernelGGL((batch_matvec_exchange_kernel<FMT, WN>), grid, dim3(64 * MV_WAVES), 0, s, w, x, y, batch,
                       static_cast<int>(rows), static_cast<int>(cols), row_bytes(FMT, cols), control);
}

// 32 rows a workgroup (x is exchanged once for both tiles) where that still
// gives every second CU one (F16 16384 x 3072 25.5 us, 30.8 with 16 rows).
template <int FMT>
hipError_t launch_rows(const uint8_t* w, const float* x, float* y, int batch, int64_t rows, int64_t cols,
                       const int32_t* control, hipStream_t s)
{
    if ((rows + 31) / 32 >= 128)
        launch_tile<FMT, 2>(w, x, y, batch, rows, cols, control, s);
    else
        launch_tile<FMT, 1>(w, x, y, batch, rows, cols, control, s);
    return hipGetLastError();
}

}  // namespace

hipError_t launch_batch_matvec_exchange(int fmt, const void* w, const float* x, float* y, int batch, int64_t rows,
                                        int64_t cols, const int32_t* control, hipStream_t s)
{
    const uint8_t* wb = static_cast<const uint8_t*>(w);
    switch (fmt) {
    case FMT_F16: return launch_rows<FMT_F16>(wb, x, y, batch, rows, cols, control, s);
    case FMT_F32: return launch_rows<FMT_F32>(wb, x, y, batch, rows, cols, control, s);
    default: return hipErrorInvalidValue;
    }
}

}  // namespace si
