// Batched prefill product Y[m, n] = sum_k X[m, k] * W[n, k] for grids that the
// LDS-tiled kernels (si_prefill.hip) cannot fill the chip with: few tokens,
// or few rows of W.
//
// A workgroup of 8 waves owns 16 * WN rows of W and 16 * MT tokens (at most
// 64); its waves split the 64-column steps of K (a contiguous run each) and share nothing until their tiles meet in LDS at the end, in wave
// order, so there is no barrier in the loop and results are reproducible.
// v_mfma_f32_16x16x32_bf16 takes its columns in any order as long as both
// operands agree, so lane (r, g) = (l % 16, l / 16) multiplies the 16 values
// of item g % 2 of block g / 2 of the step (half a 32-value block of row r:
// one 8- or 16-byte load and the block's scale), decoded straight into the
// two B fragments, with the same 16 columns of each token tile (two 16-byte A
// fragments).  Loaded by those lanes, though, neighbouring lanes would read
// different rows, and the address unit takes such a load at about one lane a
// cycle (Q8_0 3072 x 8192 at 33 tokens: 34 us).  So lane l loads row l / 4's
// item l % 4 (four neighbours share a line) and the lanes exchange through the
// wave's own part of LDS, 16-byte slots permuted so that neither side has
// bank conflicts.  Both operands are requested D steps ahead (three steps
// ahead measured no faster than two).
//
// Bound: the serial chain of a wave's steps (load, exchange, decode, two
// products per tile) on two waves a SIMD: half of it is waiting, and no unit is
// busy for more than 0.6 of the time (address unit 0.3 to 0.6, VALU 0.14 to
// 0.27, matrix cores 0.05 to 0.10).  The four projections of a 3072-wide layer (qkv, o, gate/up, down),
// Q8_0 at 33 tokens: 33.6 + 33.5 + 48.4 + 37.9 us with the LDS-tiled kernels,
// 11.8 + 8.5 + 27.8 + 21.3 us here (161 -> 76 us in one plan); 3072 x 3072 Q4_K at 1 token 29.9 -> 5.6 us,
// F16 300 x 3072 at 16 51.6 -> 5.0 us.
#include "si_prefill.hpp"
#include "si_prefill_units.hpp"

namespace si {
namespace {

constexpr int SK_WAVES = 8;

template <int FMT, int MT, int WN>
__global__ __launch_bounds__(64 * SK_WAVES) void prefill_skinny_kernel(const uint8_t* __restrict__ W,
                                                                       const __bf16* __restrict__ X,
                                                                       float* __restrict__ Y, int M, int N, int K,
                                                                       int64_t row_bytes, bool tokens_first)
{
    constexpr int D = 2;                                  // steps in flight
    constexpr int RW = FMT == FMT_Q4_0 ? 3 : FMT == FMT_Q8_0 ? 5 : FMT == FMT_F32 ? 16 : 8;   // words of an item
    constexpr int QW = RW / 4, TW = RW % 4;               // as single words, then 16-byte groups
    constexpr int GROUPS = 2 * MT + QW * WN;              // 1 KB groups of a step
    constexpr int WAVE_WORDS = 256 * GROUPS + 64 * TW * WN;
    constexpr int RED_WORDS = SK_WAVES * MT * WN * 256;
    constexpr int POOL = SK_WAVES * WAVE_WORDS > RED_WORDS ? SK_WAVES * WAVE_WORDS : RED_WORDS;
    __shared__ __attribute__((aligned(16))) uint32_t pool[POOL];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int n0 = (tokens_first ? blockIdx.y : blockIdx.x) * 16 * WN;
    const int m0 = (tokens_first ? blockIdx.x : blockIdx.y) * 16 * MT;
    const int nblk = K / 32;
    const int steps = (nblk + 1) / 2;
    const int per = (steps + SK_WAVES - 1) / SK_WAVES;
    const int s0 = wave * per, mine = min(per, steps - s0);   // this wave's steps s0 .. s0 + mine - 1 (may be none)

    // what the lane loads: item h of block bo of row lr; and what it
    // multiplies: item fg & 1 of block fg >> 1 of row fr
    const int lr = lane >> 2, bo = (lane >> 1) & 1, h = lane & 1;
    const int fr = lane & 15, fg = lane >> 4;
    uint32_t* const mine_lds = pool + wave * WAVE_WORDS;
    const int wslot = 4 * lr + ((lane & 3) ^ ((lr >> 2) & 3)), rslot = 4 * fr + (fg ^ ((fr >> 2) & 3));
    // columns of the two fragments inside a block: Q4_0 keeps elements 8h..
    // and 16 + 8h.. in one byte's nibbles
    const int c0 = FMT == FMT_Q4_0 ? 8 * h : 16 * h;   // the second fragment 16 or 8 columns on
    // lane offsets of a step (rows and tokens past the end repeat the last;
    // their results are dropped)
    uint32_t woff[WN], qoff[WN], xoff[MT];
#pragma unroll
    for (int j = 0; j < WN; j++) {
        const uint32_t row = static_cast<uint32_t>(min(n0 + 16 * j + lr, N - 1)) * static_cast<uint32_t>(row_bytes);
        woff[j] = item_off<FMT>(row, bo);
        qoff[j] = item_qoff<FMT>(row, bo, h);
    }
#pragma unroll
    for (int t = 0; t < MT; t++)
        xoff[t] = static_cast<uint32_t>(min(m0 + 16 * t + lr, M - 1)) * static_cast<uint32_t>(2 * K) + 2 * (32 * bo + c0);
    const uint8_t* const xb = reinterpret_cast<const uint8_t*>(X);
    // an odd row of blocks: the last step's second block does not exist, its
    // lanes re-read the first one's and multiply 0 by 0
    const bool odd = (nblk & 1) != 0 && s0 + mine == steps;

    f32x4 acc[MT][WN];
#pragma unroll
    for (int i = 0; i < MT; i++)
#pragma unroll
        for (int j = 0; j < WN; j++)
            acc[i][j] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};

    RawW<FMT> raw[D][WN];
    u32x4 xa[D][MT][2];
    auto load_step = [&](int k, RawW<FMT> (&wd)[WN], u32x4 (&xd)[MT][2]) {
        const int st = s0 + k;
        const uint8_t* wbase = step_base<FMT, 2>(W, st);
        const uint8_t* qbase = step_qbase<FMT, 2>(wbase, st);
        const uint8_t* xbase = xb + static_cast<int64_t>(st) * 128;
        const uint32_t back = odd && k == mine - 1 ? bo : 0;
        const uint32_t wback = FMT == FMT_Q4_K ? 0 : back * blk_bytes<FMT>();
#pragma unroll
        for (int j = 0; j < WN; j++)
            wd[j] = load_item<FMT>(wbase, qbase, woff[j] - wback, qoff[j] - wback);
#pragma unroll
        for (int t = 0; t < MT; t++) {
            const uint32_t o = opaque(xoff[t] - 64 * back);
            xd[t][0] = *reinterpret_cast<const u32x4*>(xbase + o);
            xd[t][1] = *reinterpret_cast<const u32x4*>(xbase + o + 2 * (FMT == FMT_Q4_0 ? 16 : 8));
        }
    };
    // the wave's step into its part of LDS, and its fragments out of it (a
    // wave's LDS accesses execute in order: the fences only keep the
    // compiler's order)
    auto stage = [&](const RawW<FMT> (&wd)[WN], const u32x4 (&xd)[MT][2]) {
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
        u32x4* g4 = reinterpret_cast<u32x4*>(mine_lds);
#pragma unroll
        for (int t = 0; t < MT; t++) {
            g4[64 * (2 * t) + wslot] = xd[t][0];
            g4[64 * (2 * t + 1) + wslot] = xd[t][1];
        }
#pragma unroll
        for (int j = 0; j < WN; j++) {
#pragma unroll
            for (int q = 0; q < QW; q++)
                g4[64 * (2 * MT + QW * j + q) + wslot] =
                    u32x4{wd[j].w[TW + 4 * q], wd[j].w[TW + 4 * q + 1], wd[j].w[TW + 4 * q + 2], wd[j].w[TW + 4 * q + 3]};
#pragma unroll
            for (int q = 0; q < TW; q++)
                mine_lds[256 * GROUPS + 64 * (TW * j + q) + lane] = wd[j].w[q];
        }
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
    };
    auto fetch = [&](RawW<FMT> (&wd)[WN], u32x4 (&xd)[MT][2]) {
        const u32x4* g4 = reinterpret_cast<const u32x4*>(mine_lds);
#pragma unroll
        for (int j = 0; j < WN; j++) {
#pragma unroll
            for (int q = 0; q < TW; q++)
                wd[j].w[q] = mine_lds[256 * GROUPS + 64 * (TW * j + q) + 4 * fr + fg];
#pragma unroll
            for (int q = 0; q < QW; q++) {
                const u32x4 v = g4[64 * (2 * MT + QW * j + q) + rslot];
#pragma unroll
                for (int k = 0; k < 4; k++)
                    wd[j].w[TW + 4 * q + k] = v[k];
            }
        }
#pragma unroll
        for (int t = 0; t < MT; t++) {
            xd[t][0] = g4[64 * (2 * t) + rslot];
            xd[t][1] = g4[64 * (2 * t + 1) + rslot];
        }
    };
    auto multiply = [&](int i, const RawW<FMT> (&wr)[WN], const u32x4 (&xr)[MT][2]) {
        bf16x8 b0[WN], b1[WN], a0[MT], a1[MT];
#pragma unroll
        for (int j = 0; j < WN; j++) {
            int d0, d1;
            decode_raw<FMT>(wr[j], 2 * (s0 + i) + (fg >> 1), fg & 1, b0[j], b1[j], d0, d1);
        }
#pragma unroll
        for (int t = 0; t < MT; t++) {
            a0[t] = __builtin_bit_cast(bf16x8, xr[t][0]);
            a1[t] = __builtin_bit_cast(bf16x8, xr[t][1]);
        }
        if (odd && i == mine - 1) {
            if (fg >> 1) {
#pragma unroll
                for (int j = 0; j < WN; j++)
                    b0[j] = b1[j] = bf16x8{};
#pragma unroll
                for (int t = 0; t < MT; t++)
                    a0[t] = a1[t] = bf16x8{};
            }
        }
#pragma unroll
        for (int t = 0; t < MT; t++)
#pragma unroll
            for (int j = 0; j < WN; j++)
                acc[t][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a0[t], b0[j], acc[t][j], 0, 0, 0);
#pragma unroll
        for (int t = 0; t < MT; t++)
#pragma unroll
            for (int j = 0; j < WN; j++)
                acc[t][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a1[t], b1[j], acc[t][j], 0, 0, 0);
    };
    // step i (its fragments are in LDS): the next step takes its place there
    // and the one D further is requested, into the registers that frees
    auto run_step = [&](int i, RawW<FMT> (&wn)[WN], u32x4 (&xn)[MT][2], bool next, bool more) {
        RawW<FMT> wf[WN];
        u32x4 xf[MT][2];
        fetch(wf, xf);
        if (next)
            stage(wn, xn);
        if (more)
            load_step(i + 1 + D, wn, xn);
        multiply(i, wf, xf);
    };

    if (mine > 0) {
#pragma unroll
        for (int u = 0; u < D; u++)
            load_step(min(u, mine - 1), raw[u], xa[u]);
        stage(raw[0], xa[0]);
        if (D < mine)
            load_step(D, raw[0], xa[0]);
        int i = 0;
        for (; i + 2 * D < mine; i += D) {
#pragma unroll
            for (int u = 0; u < D; u++)
                run_step(i + u, raw[(u + 1) % D], xa[(u + 1) % D], true, true);
        }
#pragma unroll
        for (int u = 0; u < 2 * D; u++)
            if (i + u < mine)
                run_step(i + u, raw[(u + 1) % D], xa[(u + 1) % D], i + u + 1 < mine, i + u + 1 + D < mine);
    }

    // the waves' tiles meet in LDS, in wave order; tile q = (t, j) is summed
    // and stored by wave q % 8
    __syncthreads();
    f32x4* red = reinterpret_cast<f32x4*>(pool);
#pragma unroll
    for (int t = 0; t < MT; t++)
#pragma unroll
        for (int j = 0; j < WN; j++)
            red[(wave * MT * WN + t * WN + j) * 64 + lane] = acc[t][j];
    __syncthreads();
    for (int q = wave; q < MT * WN; q += SK_WAVES) {
        f32x4 v = red[q * 64 + lane];
#pragma unroll
        for (int w = 1; w < SK_WAVES; w++)
            v += red[(w * MT * WN + q) * 64 + lane];
        const int n = n0 + 16 * (q % WN) + fr;
#pragma unroll
        for (int e = 0; e < 4; e++) {
            const int m = m0 + 16 * (q / WN) + 4 * fg + e;
            if (m < M && n < N)
                Y[static_cast<int64_t>(m) * N + n] = v[e];
        }
    }
}

// Consecutive workgroups go to the chip's 8 dies in turn, each with its own L2:
// the operand whose tiles they step through is read once, the other by every
// die, so the larger one is stepped through (stepping through W always, Q4_0
// 128 x 8192 at 2048 tokens 38.7 us, 18.5 now; 256 x 8192 40.6 and 24.9; the
// LDS-tiled kernels 32.7 and 34.7).
template <int FMT, int MT, int WN>
hipError_t launch_tile(const void* w, const void* x, float* y, int64_t m, int64_t n, int64_t k, hipStream_t s)
{
    const unsigned tn = static_cast<unsigned>((n + 16 * WN - 1) / (16 * WN)), tm = static_cast<unsigned>((m + 16 * MT - 1) / (16 * MT));
    const int64_t rb = row_bytes(FMT, k);
    const bool tokens_first = 2 * m * k > n * rb;
    hipLaunchKernelGGL((prefill_skinny_kernel<FMT, MT, WN>), tokens_first ? dim3(tm, tn) : dim3(tn, tm),
                       dim3(64 * SK_WAVES), 0, s, static_cast<const uint8_t*>(w), static_cast<const __bf16*>(x), y,
                       static_cast<int>(m), static_cast<int>(n), static_cast<int>(k), rb, tokens_first);
    return hipGetLastError();
}

template <int FMT, int WN>
hipError_t launch_rows(const void* w, const void* x, float* y, int64_t m, int64_t n, int64_t k, hipStream_t s)
{
    // the fewest token tiles of 64, evenly filled
    const int64_t tiles = (m + 63) / 64;
    switch ((m + 16 * tiles - 1) / (16 * tiles)) {
    case 1: return launch_tile<FMT, 1, WN>(w, x, y, m, n, k, s);
    case 2: return launch_tile<FMT, 2, WN>(w, x, y, m, n, k, s);
    case 3: return launch_tile<FMT, 3, WN>(w, x, y, m, n, k, s);
    default: return launch_tile<FMT, 4, WN>(w, x, y, m, n, k, s);
    }
}

template <int FMT>
hipError_t launch_fmt(const void* w, const void* x, float* y, int64_t m, int64_t n, int64_t k, hipStream_t s)
{
    // 32 rows a workgroup (each X fragment used twice) where that halves the
    // rounds of one workgroup per CU
    auto rounds = [&](int64_t rows) { return ((n + rows - 1) / rows * ((m + 63) / 64) + 255) / 256; };
    return rounds(32) < rounds(16) ? launch_rows<FMT, 2>(w, x, y, m, n, k, s) : launch_rows<FMT, 1>(w, x, y, m, n, k, s);
}

}  // namespace

hipError_t launch_prefill_skinny(int fmt, const void* w, const void* x_bf16, float* y, int64_t m, int64_t rows,
                                 int64_t cols, hipStream_t s)
{
    switch (fmt) {
    case FMT_Q8_0: return launch_fmt<FMT_Q8_0>(w, x_bf16, y, m, rows, cols, s);
    case FMT_Q4_0: return launch_fmt<FMT_Q4_0>(w, x_bf16, y, m, rows, cols, s);
    case FMT_Q4_K: return launch_fmt<FMT_Q4_K>(w, x_bf16, y, m, rows, cols, s);
    case FMT_F16: return launch_fmt<FMT_F16>(w, x_bf16, y, m, rows, cols, s);
    case FMT_F32: return launch_fmt<FMT_F32>(w, x_bf16, y, m, rows, cols, s);
    default: return hipErrorInvalidValue;
    }
}

}  // namespace si
