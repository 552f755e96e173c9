// Parts of the prefill products: the W decode of si_prefill.hip and
// si_prefill_skinny.hip (the raw words of 16 values of a weight row and their
// exact values rounded to bf16), and the vector types and word helpers that
// si_batch_matvec.hip uses too.
#pragma once

#include "si_internal.hpp"

#include <hip/hip_fp16.h>

namespace si {
namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));   // 16 raw bytes

// Raw words of one item of 16 values (half a 32-value block of one W row),
// loaded steps ahead of their decode.  Loads of up to 16 bytes bring whole
// words and every bit extraction happens at decode time, so a word in flight is
// never touched before its decode.  An F32 item is 16 words, every other format's
// at most 8.
template <int FMT>
struct RawW {
    uint32_t w[FMT == FMT_F32 ? 16 : 8];
};

// 16 or 8 bytes at a 2-byte aligned address, one load.
struct __attribute__((packed, aligned(2))) words4_a2 {
    uint32_t w[4];
};
struct __attribute__((packed, aligned(2))) words2_a2 {
    uint32_t w[2];
};

__device__ __forceinline__ uint32_t ld_u16(const uint8_t* p)
{
    return *reinterpret_cast<const unsigned short*>(p);
}

// Hides a value from the optimiser: keeps a 32-bit lane offset from being
// widened to 64 bits outside the loop (so loads keep the scalar-base
// addressing form), and keeps the known-zero bits of a masked word hidden
// (so each byte converts with one v_cvt_f32_ubyteN).
__device__ __forceinline__ uint32_t opaque(uint32_t v)
{
    asm("" : "+v"(v));
    return v;
}

// Bytes of a 32-column block of a row (Q4_K super-blocks are addressed apart).
template <int FMT>
constexpr int blk_bytes() { return FMT == FMT_Q4_0 ? 18 : FMT == FMT_Q8_0 ? 34 : FMT == FMT_F16 ? 64 : 128; }

// A step is BPS (2 or 4) blocks of every row, from a multiple of BPS on.  Its
// uniform base: the rows' bytes of the step (Q4_K: of its super-block), and
// for Q4_K the step's first chunk of quant bytes.
template <int FMT, int BPS>
__device__ __forceinline__ const uint8_t* step_base(const uint8_t* W, int step)
{
    return W + (FMT == FMT_Q4_K ? static_cast<int64_t>((BPS * step) >> 3) * 144
                                : static_cast<int64_t>(step) * (BPS * blk_bytes<FMT>()));
}
template <int FMT, int BPS>
__device__ __forceinline__ const uint8_t* step_qbase(const uint8_t* base, int step)
{
    return FMT == FMT_Q4_K ? base + 16 + 32 * (((BPS * step) & 7) >> 1) : base;
}
// A lane's 32-bit offsets from those: block bo (< BPS) of the row at row_off,
// and item h's quant bytes in it.
template <int FMT>
__device__ __forceinline__ uint32_t item_off(uint32_t row_off, int bo)
{
    return row_off + (FMT == FMT_Q4_K ? 0 : blk_bytes<FMT>() * bo);
}
template <int FMT>
__device__ __forceinline__ uint32_t item_qoff(uint32_t row_off, int bo, int h)
{
    return FMT == FMT_Q4_K ? row_off + 32 * (bo >> 1) + 16 * h
                           : item_off<FMT>(row_off, bo) +
                                 (FMT == FMT_Q4_0 ? 2 + 8 * h : FMT == FMT_Q8_0 ? 2 + 16 * h : blk_bytes<FMT>() / 2 * h);
}

// Item h of a block, with the widest loads the layout allows (one load
// instruction costs the address unit about a cycle per four lanes of a row
// whatever its width: loaded word by word, Q4_K items took twice the
// matrix-core time of a step; the four projections of a 3072-wide layer at 2048
// tokens 794 -> 551 us) and no vector address arithmetic:
//   Q4_0 {fp16 d; u8 qs[16]}: d and bytes 8h..8h+7 (elements 8h..8h+7 in the
//        low nibbles, 16+8h..16+8h+7 in the high nibbles);
//   Q8_0 {fp16 d; int8 q[32]}: d and q[16h..16h+15];
//   Q4_K {fp16 d, dmin; u8 scales[12]; u8 qs[128]}, sub-block j = blk % 8:
//        d | dmin << 16, the three scale words and the 16 quant bytes of
//        elements 16h..16h+15 (nibble j % 2 of qs[32 (j / 2) + 16h ..]);
//   F16 / F32: elements 16h..16h+15, 8 or 16 words.
template <int FMT>
__device__ __forceinline__ RawW<FMT> load_item(const uint8_t* base, const uint8_t* qbase, uint32_t off, uint32_t qoff)
{
    RawW<FMT> r;
    off = opaque(off);
    qoff = opaque(qoff);
    if constexpr (FMT == FMT_Q4_0) {
        r.w[0] = ld_u16(base + off);
        const words2_a2 q = *reinterpret_cast<const words2_a2*>(base + qoff);
        r.w[1] = q.w[0]; r.w[2] = q.w[1];
    } else if constexpr (FMT == FMT_Q8_0) {
        r.w[0] = ld_u16(base + off);
        const words4_a2 q = *reinterpret_cast<const words4_a2*>(base + qoff);
        r.w[1] = q.w[0]; r.w[2] = q.w[1]; r.w[3] = q.w[2]; r.w[4] = q.w[3];
    } else if constexpr (FMT == FMT_Q4_K) {
        const words4_a2 hd = *reinterpret_cast<const words4_a2*>(base + off);
        const words4_a2 q = *reinterpret_cast<const words4_a2*>(qbase + qoff);
#pragma unroll
        for (int k = 0; k < 4; k++) {
            r.w[k] = hd.w[k];
            r.w[4 + k] = q.w[k];
        }
    } else {
#pragma unroll
        for (int i = 0; i < (FMT == FMT_F16 ? 2 : 4); i++) {
            const words4_a2 q = *reinterpret_cast<const words4_a2*>(base + qoff + 16 * i);
#pragma unroll
            for (int k = 0; k < 4; k++)
                r.w[4 * i + k] = q.w[k];
        }
    }
    return r;
}

__device__ __forceinline__ float half_bits(uint32_t h)
{
    return __half2float(__ushort_as_half(static_cast<unsigned short>(h & 0xffffu)));
}

// Byte i of q as a float (v_cvt_f32_ubyteN).
__device__ __forceinline__ float ubyte(uint32_t q, int i) { return static_cast<float>((q >> (8 * i)) & 0xffu); }

// 8 values fma(a, byte, c) of two words, rounded to bf16 (RNE).
__device__ __forceinline__ bf16x8 decode8(uint32_t q0, uint32_t q1, float a, float c)
{
    f32x8 v;
#pragma unroll
    for (int i = 0; i < 4; i++) {
        v[i] = fmaf(a, ubyte(q0, i), c);
        v[4 + i] = fmaf(a, ubyte(q1, i), c);
    }
    return __builtin_convertvector(v, bf16x8);
}

// The 16 values of an item in FP32 are bit-identical to the block decoder,
// each one fused multiply-add whose exact result needs no rounding or
// equals the decoder's single rounding:
//   Q8_0: d * q = fma(d, q + 128, -128 d)   (d * (q + 128) and 128 d exact)
//   Q4_0: d * (q - 8) = fma(d, q, -8 d)      (every term exact)
//   Q4_K: (d sc) q - dmin m = fma(d1, q, -m1) with d1 = d sc and m1 = dmin m
//         exact (11-bit by 6-bit products), d1 q exact, one rounding.
// High nibbles are masked in place (16 q per byte) and the factor 1/16 goes
// into the scale, which stays exact (a power of two).  The two halves of
// 8 values go to columns c0 and c1 of the block.
template <int FMT>
__device__ __forceinline__ void decode_raw(const RawW<FMT>& r, int blk, int h, bf16x8& v0, bf16x8& v1, int& c0,
                                           int& c1);

template <>
__device__ __forceinline__ void decode_raw<FMT_Q4_0>(const RawW<FMT_Q4_0>& r, int, int h, bf16x8& v0, bf16x8& v1, int& c0,
                                                     int& c1)
{
    const float d = half_bits(r.w[0]);
    const float c = -8.0f * d;
    v0 = decode8(opaque(r.w[1] & 0x0f0f0f0fu), opaque(r.w[2] & 0x0f0f0f0fu), d, c);
    v1 = decode8(opaque(r.w[1] & 0xf0f0f0f0u), opaque(r.w[2] & 0xf0f0f0f0u), d * 0.0625f, c);
    c0 = 8 * h;
    c1 = 16 + 8 * h;
}

template <>
__device__ __forceinline__ void decode_raw<FMT_Q8_0>(const RawW<FMT_Q8_0>& r, int, int h, bf16x8& v0, bf16x8& v1, int& c0,
                                                     int& c1)
{
    const float d = half_bits(r.w[0]);
    const float c = -128.0f * d;
    v0 = decode8(opaque(r.w[1] ^ 0x80808080u), opaque(r.w[2] ^ 0x80808080u), d, c);   // q + 128 as unsigned bytes
    v1 = decode8(opaque(r.w[3] ^ 0x80808080u), opaque(r.w[4] ^ 0x80808080u), d, c);
    c0 = 16 * h;
    c1 = 16 * h + 8;
}

// 6-bit scale and min of sub-block j (GGML get_scale_min_k4) from the
// scale words lo = scales[0..3], mid = scales[4..7], hi = scales[8..11].
template <>
__device__ __forceinline__ void decode_raw<FMT_Q4_K>(const RawW<FMT_Q4_K>& r, int blk, int h, bf16x8& v0, bf16x8& v1, int& c0,
                                                     int& c1)
{
    const int j = blk & 7;
    const float d = half_bits(r.w[0]), dmin = half_bits(r.w[0] >> 16);
    const int sh = 8 * (j & 3);
    const uint32_t lo = (r.w[1] >> sh) & 0xffu, mid = (r.w[2] >> sh) & 0xffu, hi = (r.w[3] >> sh) & 0xffu;
    int sc, m;
    if (j < 4) {
        sc = static_cast<int>(lo & 63u);
        m = static_cast<int>(mid & 63u);
    } else {
        sc = static_cast<int>((hi & 15u) | ((lo >> 6) << 4));
        m = static_cast<int>((hi >> 4) | ((mid >> 6) << 4));
    }
    const float d1 = __fmul_rn(d, static_cast<float>(sc));
    const float m1 = __fmul_rn(dmin, static_cast<float>(m));
    const bool high = (j & 1) != 0;
    const uint32_t mask = high ? 0xf0f0f0f0u : 0x0f0f0f0fu;
    const float a = high ? d1 * 0.0625f : d1;
    v0 = decode8(opaque(r.w[4] & mask), opaque(r.w[5] & mask), a, -m1);
    v1 = decode8(opaque(r.w[6] & mask), opaque(r.w[7] & mask), a, -m1);
    c0 = 16 * h;
    c1 = 16 * h + 8;
}

// F16: each value converted exactly to FP32, then rounded to bf16 (one
// rounding from the exact value).  F32: rounded to bf16.
template <>
__device__ __forceinline__ void decode_raw<FMT_F16>(const RawW<FMT_F16>& r, int, int h, bf16x8& v0, bf16x8& v1,
                                                    int& c0, int& c1)
{
    f32x8 a, b;
#pragma unroll
    for (int i = 0; i < 4; i++) {
        a[2 * i] = half_bits(r.w[i]);
        a[2 * i + 1] = half_bits(r.w[i] >> 16);
        b[2 * i] = half_bits(r.w[4 + i]);
        b[2 * i + 1] = half_bits(r.w[4 + i] >> 16);
    }
    v0 = __builtin_convertvector(a, bf16x8);
    v1 = __builtin_convertvector(b, bf16x8);
    c0 = 16 * h;
    c1 = 16 * h + 8;
}

template <>
__device__ __forceinline__ void decode_raw<FMT_F32>(const RawW<FMT_F32>& r, int, int h, bf16x8& v0, bf16x8& v1,
                                                    int& c0, int& c1)
{
    f32x8 a, b;
#pragma unroll
    for (int i = 0; i < 8; i++) {
        a[i] = __uint_as_float(r.w[i]);
        b[i] = __uint_as_float(r.w[8 + i]);
    }
    v0 = __builtin_convertvector(a, bf16x8);
    v1 = __builtin_convertvector(b, bf16x8);
    c0 = 16 * h;
    c1 = 16 * h + 8;
}

}  // namespace
}  // namespace si
