// Device and host parts shared by the matrix-vector kernels (si_gemv.hip,
// si_gemv_stream.hip): block decoders of a lane's unit of weights, launch
// descriptors, output functions.
#pragma once

#include "si_gemv.hpp"
#include "si_internal.hpp"
#include "si_lanes.hpp"
#include "si_planes.hpp"

#include <hip/hip_fp16.h>

#include <algorithm>

namespace si {
namespace {


constexpr int WG = 256;          // threads per workgroup (4 waves)
constexpr int XS_UNIT = 68;      // LDS floats per unit: 64 values + 4 pad (bank spread)

struct __attribute__((aligned(4))) u32x4 {
    uint32_t x, y, z, w;
};

__device__ __forceinline__ u32x4 ld4(const uint8_t* p) { return *reinterpret_cast<const u32x4*>(p); }
__device__ __forceinline__ uint32_t ld1(const uint8_t* p) { return *reinterpret_cast<const uint32_t*>(p); }

__device__ __forceinline__ float half_lo(uint32_t v)
{
    return __half2float(__ushort_as_half(static_cast<unsigned short>(v & 0xffffu)));
}
__device__ __forceinline__ float half_hi(uint32_t v)
{
    return __half2float(__ushort_as_half(static_cast<unsigned short>(v >> 16)));
}

// Sum of v over the wave, in every lane: DPP inside each 16-lane row, then
// swaps between the halves and between row pairs.
__device__ __forceinline__ float wave_sum(float v);

// 4 signed bytes of q times 4 floats, accumulated.
__device__ __forceinline__ float dot4_i8(uint32_t q, const float4& x, float a)
{
    a = fmaf(static_cast<float>(static_cast<int8_t>(q)), x.x, a);
    a = fmaf(static_cast<float>(static_cast<int8_t>(q >> 8)), x.y, a);
    a = fmaf(static_cast<float>(static_cast<int8_t>(q >> 16)), x.z, a);
    a = fmaf(static_cast<float>(static_cast<int8_t>(q >> 24)), x.w, a);
    return a;
}

// Hides the known-zero bits of a masked value from the optimiser, so the
// byte conversions below select one v_cvt_f32_ubyteN each instead of a
// bit-field extract plus a conversion.
__device__ __forceinline__ uint32_t opaque(uint32_t v)
{
    asm("" : "+v"(v));
    return v;
}

// Sum of v over aligned groups of N lanes (N = 2, 4, 8, 16), left in every
// lane of the group, with DPP lane moves (no LDS traffic):
// xor-1 and xor-2 swaps inside quads, then the mirror of each 8- and
// 16-lane row, which pairs every lane with one in the other half.
template <int N>
__device__ __forceinline__ float group_sum(float v)
{
    if constexpr (N >= 2)
        v += dpp_row<0xB1>(v);   // quad_perm 1,0,3,2
    if constexpr (N >= 4)
        v += dpp_row<0x4E>(v);   // quad_perm 2,3,0,1
    if constexpr (N >= 8)
        v += dpp_row<0x141>(v);  // row_half_mirror
    if constexpr (N >= 16)
        v += dpp_row<0x140>(v);  // row_mirror
    static_assert(N <= 16, "groups wider than a DPP row use shuffles");
    return v;
}

// ---- x as integer digit planes ----------------------------------------------
// The staged x of the 4-bit formats (and of Q8_0 at some shapes) is held as
// int8 digit planes (encode_planes: a power-of-two scale per 32-column
// block, x rounded to a 21-bit grid, at most 2^-21 M per value for a block
// of largest magnitude M).  The FP32 reference multiplies the FP32 x itself
// (CpuHalfMatrixOperators.cs:29-41); the products' error stays within the
// mat-vec tolerance but is not the reference's FP32 rounding.  Per block
// and row the planes' products combine in INT32 and the block enters the
// FP32 row sum once: d * 2^-s * sum((q - offset) * X).
//
// LDS per 64-column unit (PLANE_UNIT words): block h's planes at 24h +
// 8p + w (word w = values 4w..4w+3 of the block), then inv_0, inv_1
// (2^-s, or NaN when the block takes the per-weight FP32 form with x read
// from global memory), then aux_0, aux_1 (Q4_0: 8 sum(X) as INT32; Q4_K:
// sum(X) 2^-s as FP32; unused by Q8_0).  52 words: 16 lanes reading
// consecutive units with 16-byte reads touch distinct banks.
constexpr int PLANE_UNIT = 52;

__device__ __forceinline__ float wave_sum(float v)
{
    v = group_sum<16>(v);
    const auto a = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    v = __uint_as_float(a[0]) + __uint_as_float(a[1]);
    const auto b = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    return __uint_as_float(b[0]) + __uint_as_float(b[1]);
}

// 4 unsigned bytes (each < 256) of q times 4 floats, accumulated.
__device__ __forceinline__ float dot4_u8(uint32_t q, const float4& x, float a)
{
    a = fmaf(static_cast<float>(q & 0xffu), x.x, a);
    a = fmaf(static_cast<float>((q >> 8) & 0xffu), x.y, a);
    a = fmaf(static_cast<float>((q >> 16) & 0xffu), x.z, a);
    a = fmaf(static_cast<float>(q >> 24), x.w, a);
    return a;
}

template <int FMT>
struct QUnit;

// Two Q8_0 blocks {fp16 d; int8 q[32]} back to back.
template <>
struct QUnit<FMT_Q8_0> {
    static constexpr int UNIT_BYTES = 68;
    uint32_t v[17];
    __device__ __forceinline__ void prepare() {}

    __device__ __forceinline__ void load(const uint8_t* row, int u)
    {
        const uint8_t* p = row + u * UNIT_BYTES;
        const u32x4 a = ld4(p), b = ld4(p + 16), c = ld4(p + 32), d = ld4(p + 48);
        v[0] = a.x; v[1] = a.y; v[2] = a.z; v[3] = a.w;
        v[4] = b.x; v[5] = b.y; v[6] = b.z; v[7] = b.w;
        v[8] = c.x; v[9] = c.y; v[10] = c.z; v[11] = c.w;
        v[12] = d.x; v[13] = d.y; v[14] = d.z; v[15] = d.w;
        v[16] = ld1(p + 64);
    }

    // Contribution of block h (columns 32h..32h+31 of the unit).
    __device__ __forceinline__ float half(int h, const float4* x, float /*sx*/) const
    {
        float a0 = 0.0f, a1 = 0.0f;
#pragma unroll
        for (int k = 0; k < 8; k += 2) {
            const uint32_t q0 = h == 0 ? __builtin_amdgcn_alignbit(v[k + 1], v[k], 16) : v[9 + k];
            const uint32_t q1 = h == 0 ? __builtin_amdgcn_alignbit(v[k + 2], v[k + 1], 16) : v[10 + k];
            a0 = dot4_i8(q0, x[k], a0);
            a1 = dot4_i8(q1, x[k + 1], a1);
        }
        const float d = h == 0 ? half_lo(v[0]) : half_hi(v[8]);
        return d * (a0 + a1);
    }

    // Block h against x's digit planes P; inv = 2^-s.  sum(q X) scaled by
    // 2^-s (exact) and by the block scale, as the per-weight form
    // d * sum(q x) does.
    __device__ __forceinline__ float planes(int h, const uint32_t* P, float inv, float /*aux*/, float acc) const
    {
        uint32_t q[8];
#pragma unroll
        for (int k = 0; k < 8; k++)
            q[k] = h == 0 ? __builtin_amdgcn_alignbit(v[k + 1], v[k], 16) : v[9 + k];
        const float d = h == 0 ? half_lo(v[0]) : half_hi(v[8]);
        return fmaf(d, q8_planes_sum(q, P) * inv, acc);
    }

    // Non-finite or huge x: the per-weight FP32 form above.
    __device__ float half_exact(int h, const float4* x) const { return half(h, x, 0.0f); }
};

// Two Q4_0 blocks {fp16 d; u8 q[16]}: element j < 16 is the low nibble of
// q[j], element j + 16 the high nibble, value d * (nibble - 8).
// Fast form: the low nibbles are masked in place (q & 0x0f..) and the high
// ones too (q & 0xf0.., i.e. 16 * nibble), each byte converted by one
// v_cvt_f32_ubyteN; the factor 16 and the offset 8 are applied once per
// block: d * (a_lo + a_hi / 16 - 8 * sum(x)).
template <>
struct QUnit<FMT_Q4_0> {
    static constexpr int UNIT_BYTES = 36;
    uint32_t v[9];
    __device__ __forceinline__ void prepare() {}

    __device__ __forceinline__ void load(const uint8_t* row, int u)
    {
        const uint8_t* p = row + u * UNIT_BYTES;
        const u32x4 a = ld4(p), b = ld4(p + 16);
        v[0] = a.x; v[1] = a.y; v[2] = a.z; v[3] = a.w;
        v[4] = b.x; v[5] = b.y; v[6] = b.z; v[7] = b.w;
        v[8] = ld1(p + 32);
    }

    __device__ __forceinline__ uint32_t qword(int h, int k) const
    {
        return h == 0 ? __builtin_amdgcn_alignbit(v[k + 1], v[k], 16) : v[5 + k];
    }
    __device__ __forceinline__ float scale(int h) const { return h == 0 ? half_lo(v[0]) : half_hi(v[4]); }

    __device__ __forceinline__ float half(int h, const float4* x, float sx) const
    {
        float a_lo = 0.0f, a_hi = 0.0f;
#pragma unroll
        for (int k = 0; k < 4; k++) {
            const uint32_t q = qword(h, k);
            a_lo = dot4_u8(opaque(q & 0x0f0f0f0fu), x[k], a_lo);
            a_hi = dot4_u8(opaque(q & 0xf0f0f0f0u), x[4 + k], a_hi);
        }
        return scale(h) * fmaf(-8.0f, sx, fmaf(a_hi, 0.0625f, a_lo));
    }

    // Block h against x's digit planes P (24 words, plane p word w at
    // 8p + w); inv = 2^-s, sum8 = 8 sum(X).  Low nibbles are values 4k..4k+3
    // (plane word k), high nibbles values 16+4k.. (word 4+k).
    __device__ __forceinline__ float planes(int h, const uint32_t* P, float inv, int sum8, float acc) const
    {
        constexpr uint32_t M = 0x0f0f0f0fu;
        uint32_t lo[4], hi[4];
#pragma unroll
        for (int k = 0; k < 4; k++) {
            if (h == 0) {
                lo[k] = __builtin_amdgcn_alignbit(v[k + 1], v[k], 16) & M;
                hi[k] = __builtin_amdgcn_alignbit(v[k + 1], v[k], 20) & M;
            } else {
                lo[k] = v[5 + k] & M;
                hi[k] = (v[5 + k] >> 4) & M;
            }
        }
        return fmaf(scale(h) * inv, static_cast<float>(q4_planes_sum(lo, hi, P) - sum8), acc);
    }

    // Classification-exact form for non-finite or huge x: (nibble ^ 8) is
    // (nibble - 8) as a signed 4-bit number; moved to the top of a byte it
    // reads as the signed byte 16 * (nibble - 8), so every product carries
    // the sign and class of the dequantised weight (no sum(x) term).
    __device__ float half_exact(int h, const float4* x) const
    {
        float a = 0.0f;
        for (int k = 0; k < 4; k++) {
            const uint32_t t = qword(h, k) ^ 0x88888888u;
            a = dot4_i8((t << 4) & 0xf0f0f0f0u, x[k], a);
            a = dot4_i8(t & 0xf0f0f0f0u, x[4 + k], a);
        }
        return (scale(h) * 0.0625f) * a;
    }
};

// Q4_K super-block {fp16 d; fp16 dmin; u8 scales[12]; u8 q[128]}; unit u is
// chunk c = u % 4 (64 elements: low nibbles of q[32c..32c+31] are sub-block
// 2c, high nibbles sub-block 2c+1), value (d*sc)*q - (dmin*m).
template <>
struct QUnit<FMT_Q4_K> {
    static constexpr int UNIT_BYTES = 36;   // amortised: 144 bytes per 4 units
    uint32_t hd[4];
    uint32_t qs[8];
    int chunk;

    __device__ __forceinline__ void load(const uint8_t* row, int u)
    {
        chunk = u & 3;
        const uint8_t* p = row + (u >> 2) * 144;
        const u32x4 h = ld4(p), a = ld4(p + 16 + 32 * chunk), b = ld4(p + 32 + 32 * chunk);
        hd[0] = h.x; hd[1] = h.y; hd[2] = h.z; hd[3] = h.w;
        qs[0] = a.x; qs[1] = a.y; qs[2] = a.z; qs[3] = a.w;
        qs[4] = b.x; qs[5] = b.y; qs[6] = b.z; qs[7] = b.w;
    }

    // d * sc and dmin * m of the unit's sub-blocks 2c (low nibbles) and
    // 2c + 1 (high nibbles), c = chunk (GGML get_scale_min_k4).  Their scale
    // bytes are the pair jj, jj + 1 with jj = 2 (c % 2) of each scale word,
    // so both are extracted at once (byte lanes of a 16-bit field), with
    // selects so lanes of different chunks do not diverge:
    //   j < 4:  sc = scales[j] & 63, m = scales[j + 4] & 63
    //   j >= 4: sc = (scales[j + 4] & 15) | (scales[j - 4] >> 6) << 4,
    //           m = (scales[j + 4] >> 4) | (scales[j] >> 6) << 4
    float dsc[2], dmn[2];
    __device__ __forceinline__ void prepare()
    {
        const int sh = 16 * (chunk & 1);
        const uint32_t s0 = hd[1] >> sh, s1 = hd[2] >> sh, s2 = hd[3] >> sh;
        const bool low = chunk < 2;
        const uint32_t sc = low ? (s0 & 0x3f3fu) : ((s2 & 0x0f0fu) | ((s0 >> 2) & 0x3030u));
        const uint32_t m = low ? (s1 & 0x3f3fu) : (((s2 >> 4) & 0x0f0fu) | ((s1 >> 2) & 0x3030u));
        const float d = half_lo(hd[0]), dm = half_hi(hd[0]);
        dsc[0] = d * static_cast<float>(sc & 0xffu);
        dsc[1] = d * static_cast<float>((sc >> 8) & 0xffu);
        dmn[0] = dm * static_cast<float>(m & 0xffu);
        dmn[1] = dm * static_cast<float>((m >> 8) & 0xffu);
    }

    // The high nibbles are masked in place (16 * q per byte); 1/16 goes
    // into the sub-block scale, which stays exact (a power of two).
    __device__ __forceinline__ float half(int h, const float4* x, float sx) const
    {
        const uint32_t mask = h == 0 ? 0x0f0f0f0fu : 0xf0f0f0f0u;
        float a0 = 0.0f, a1 = 0.0f;
#pragma unroll
        for (int k = 0; k < 8; k += 2) {
            a0 = dot4_u8(opaque(qs[k] & mask), x[k], a0);
            a1 = dot4_u8(opaque(qs[k + 1] & mask), x[k + 1], a1);
        }
        const float d1 = dsc[h] * (h == 0 ? 1.0f : 0.0625f);
        return fmaf(d1, a0 + a1, -(dmn[h] * sx));
    }

    // Sub-block 2c + h against x's digit planes P (nibble word k holds
    // values 4k..4k+3, plane word k); inv = 2^-s, sxq = sum(X) 2^-s.
    __device__ __forceinline__ float planes(int h, const uint32_t* P, float inv, float sxq, float acc) const
    {
        constexpr uint32_t M = 0x0f0f0f0fu;
        uint32_t q[8];
#pragma unroll
        for (int k = 0; k < 8; k++)
            q[k] = (h == 0 ? qs[k] : qs[k] >> 4) & M;
        int s = 0;
#pragma unroll
        for (int p = 2; p >= 0; p--) {
            if (p < 2)
                s <<= 8;
#pragma unroll
            for (int k = 0; k < 8; k++)
                s = dot4_planes(q[k], P[8 * p + k], s);
        }
        return fmaf(dsc[h] * inv, static_cast<float>(s), fmaf(-dmn[h], sxq, acc));
    }

    // Same contribution with every weight decoded as the oracle does,
    // w = (d*sc)*q - (dmin*m) rounded per operation, then w*x accumulated.
    // Used when x holds non-finite or huge values, where the factored form
    // above could change the IEEE class of the result (inf - inf).
    __device__ float half_exact(int h, const float4* x) const
    {
        const float d1 = dsc[h], m1 = dmn[h];
        float a = 0.0f;
        for (int k = 0; k < 8; k++) {
            const uint32_t q = h == 0 ? (qs[k] & 0x0f0f0f0fu) : ((qs[k] >> 4) & 0x0f0f0f0fu);
            const float xs[4] = {x[k].x, x[k].y, x[k].z, x[k].w};
            for (int i = 0; i < 4; i++) {
                const float w = __fsub_rn(__fmul_rn(d1, static_cast<float>((q >> (8 * i)) & 0xffu)), m1);
                a = fmaf(w, xs[i], a);
            }
        }
        return a;
    }
};

// 64 F16 weights (128 bytes, 32 words): each weight converted exactly to
// FP32 and multiplied into the sum in one fused op (v_fma_mix_f32), the
// reference's ConvertToSingle + Dot (CpuHalfMatrixOperators.cs:29-41).
template <>
struct QUnit<FMT_F16> {
    static constexpr int UNIT_BYTES = 128;
    uint32_t v[32];
    __device__ __forceinline__ void prepare() {}

    __device__ __forceinline__ void load(const uint8_t* row, int u)
    {
        const uint8_t* p = row + u * UNIT_BYTES;
#pragma unroll
        for (int i = 0; i < 8; i++) {
            const u32x4 a = ld4(p + 16 * i);
            v[4 * i] = a.x; v[4 * i + 1] = a.y; v[4 * i + 2] = a.z; v[4 * i + 3] = a.w;
        }
    }

    __device__ __forceinline__ float half(int h, const float4* x, float /*sx*/) const
    {
        float a0 = 0.0f, a1 = 0.0f;
#pragma unroll
        for (int k = 0; k < 8; k++) {
            const uint32_t w0 = v[16 * h + 2 * k], w1 = v[16 * h + 2 * k + 1];
            a0 = fmaf(half_lo(w0), x[k].x, a0);
            a1 = fmaf(half_hi(w0), x[k].y, a1);
            a0 = fmaf(half_lo(w1), x[k].z, a0);
            a1 = fmaf(half_hi(w1), x[k].w, a1);
        }
        return a0 + a1;
    }
};

// 64 F32 weights (256 bytes), one FMA each (CpuPrimitiveOperatorBackend.cs:222-227).
template <>
struct QUnit<FMT_F32> {
    static constexpr int UNIT_BYTES = 256;
    uint32_t v[64];
    __device__ __forceinline__ void prepare() {}

    __device__ __forceinline__ void load(const uint8_t* row, int u)
    {
        const uint8_t* p = row + u * UNIT_BYTES;
#pragma unroll
        for (int i = 0; i < 16; i++) {
            const u32x4 a = ld4(p + 16 * i);
            v[4 * i] = a.x; v[4 * i + 1] = a.y; v[4 * i + 2] = a.z; v[4 * i + 3] = a.w;
        }
    }

    __device__ __forceinline__ float half(int h, const float4* x, float /*sx*/) const
    {
        float a0 = 0.0f, a1 = 0.0f;
#pragma unroll
        for (int k = 0; k < 8; k++) {
            const uint32_t* w = v + 32 * h + 4 * k;
            a0 = fmaf(__uint_as_float(w[0]), x[k].x, a0);
            a1 = fmaf(__uint_as_float(w[1]), x[k].y, a1);
            a0 = fmaf(__uint_as_float(w[2]), x[k].z, a0);
            a1 = fmaf(__uint_as_float(w[3]), x[k].w, a1);
        }
        return a0 + a1;
    }
};

// ---- launch descriptors -----------------------------------------------------

// Device copy of one GemvOp.  A launch carries up to MAX_SEGS of them by
// value.  The tiled kernel runs a 1D grid of exactly the ops' workgroups
// (op i from workgroup first[i]; a workgroup finds its op with a uniform
// scan of the kernel arguments); the streaming, short-row and any-shape kernels
// run a 2D grid, grid row i being op i (as wide as the largest op needs), whose
// workgroups past their op's rows leave before any load or barrier.
struct Seg {
    const uint8_t* w;
    const float* x;
    float* y;
    const float* residual;
    const float* nw;        // norm weight
    const float* nb;        // norm bias
    const float* mix;
    const float* prev;
    float* norm_out;
    const float* copy_src;
    float* copy_dst;
    int rows;               // output rows
    int in;                 // XformKind
    int out;                // OutKind
    int copy_n;
    int blocks;             // blocks per row (all but the tiled kernel)
    float eps;
};
// A launch of one op carries a one-entry table, so its kernel reads its
// descriptor at fixed kernel-argument offsets (no dependent lookup).
template <int NS>
struct Segs {
    Seg s[NS];
    int count;
    // tiled kernel, NS > 1: a 1D grid, op i owning workgroups first[i] ..
    // first[i + 1] - 1 (the short-row and any-shape kernels run one grid
    // row per op instead)
    int first[NS];
};

// Output function of one row (OUT_SWIGLU_ROWS is handled by the callers,
// which hold both halves); res is the row's residual, loaded at the start
// of the kernel when the op has one.
__device__ __forceinline__ float finish(const Seg& sg, float v, float res, bool has_res)
{
    switch (sg.out) {
    case OUT_RELU_SQUARE: {
        const float h = v > 0.0f ? v : (v != v ? v : 0.0f);   // max(v, 0) with NaN kept
        return h * h;
    }
    case OUT_TANH: return tanhf(v);
    case OUT_SIGMOID: return 1.0f / (1.0f + expf(-v));
    default: return has_res ? v + res : v;
    }
}

__device__ __forceinline__ float silu_mul(float g, float u)
{
    return g / (1.0f + expf(-g)) * u;
}

// The op's first workgroup copies copy_n floats (a state store that must
// happen after every reader of the destination has run).  The first
// SIDE_HELD * threads values are loaded at the start of the kernel, ahead
// of the weights, and stored at its end; the rest (if any) at the end.
constexpr int SIDE_HELD = 8;

// The whole copy in one pass (kernels whose weight stream is short).
__device__ __forceinline__ void side_copy(const Seg& sg, int b, int threads)
{
    if (sg.copy_n > 0 && b == 0)
        for (int i = threadIdx.x; i < sg.copy_n; i += threads)
            sg.copy_dst[i] = sg.copy_src[i];
}

__device__ __forceinline__ float ld_half(const uint8_t* p)
{
    const unsigned short h = static_cast<unsigned short>(p[0] | (p[1] << 8));
    return __half2float(__ushort_as_half(h));
}

// One F16 / F32 weight from its bytes (byte loads: no alignment needs).
template <int FMT>
__device__ __forceinline__ float elem(const uint8_t* p)
{
    if constexpr (FMT == FMT_F16)
        return ld_half(p);
    return __uint_as_float(static_cast<uint32_t>(p[0]) | (static_cast<uint32_t>(p[1]) << 8) |
                           (static_cast<uint32_t>(p[2]) << 16) | (static_cast<uint32_t>(p[3]) << 24));
}

// ---- descriptor tables (host) -------------------------------------------------

inline Seg to_seg(const GemvOp& op)
{
    Seg g{};
    g.w = static_cast<const uint8_t*>(op.w);
    g.x = op.x;
    g.y = op.y;
    g.residual = op.residual;
    g.nw = op.norm_weight;
    g.nb = op.norm_bias;
    g.mix = op.mix;
    g.prev = op.prev;
    g.norm_out = op.norm_out;
    g.copy_src = op.copy_src;
    g.copy_dst = op.copy_dst;
    g.copy_n = static_cast<int>(op.copy_n);
    g.rows = static_cast<int>(op.rows);
    g.in = op.in;
    g.out = op.out;
    g.blocks = static_cast<int>(op.cols / block_elems(op.fmt));
    g.eps = op.eps;
    return g;
}

// Builds the descriptor table of n ops and returns the 2D launch grid: op
// i takes ceil(rows / per_wg(op)) workgroups; a table of several ops runs
// one grid row per op, as wide as the largest op needs.
template <int NS, typename PerWg>
dim3 fill_segs(Segs<NS>& t, const GemvOp* ops, int n, PerWg per_wg)
{
    t = Segs<NS>{};
    t.count = n;
    unsigned width = 1;
    for (int i = 0; i < n; i++) {
        t.s[i] = to_seg(ops[i]);
        const int per = per_wg(ops[i]);
        width = std::max(width, static_cast<unsigned>((ops[i].rows + per - 1) / per));
    }
    return dim3(width, static_cast<unsigned>(n));
}

}  // namespace
}  // namespace si
