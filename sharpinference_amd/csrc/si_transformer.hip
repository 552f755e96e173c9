// The transformer operators of the reference's D3D12 decode program as
// separate launches, with the reference's semantics and buffer layouts
// (SharpInference.Instructions.D3D12/GpuTransformerInstructionCollection.cs):
//
//   rms-norm            :323-368   out = x * (1 / sqrt(sum(x^2) / n + eps)) * w
//   residual-rms-norm   :370-417   updated = hidden + residual; out = rms-norm(updated)
//   swiglu              :419-443   out_i = g_i / (1 + exp(-g_i)) * u_i over [g | u]
//   rope-kv-write       :445-543   rotate q and k of one token at *position, write
//                                  q to `query` and k, v to cache row *position
//   grouped-query-attention :46-143  softmax(q . K^T / sqrt(head)) . V over rows
//                                  0..min(max(*position, 0), context - 1), split
//                                  into 64-row chunks merged by a second launch
//
// KV caches are [context][kv_heads][head_size] (a token's row holds every KV
// head), FP32 as in the reference or fp16 (rounded to nearest even on
// write).  The fused decode step (si_decode.hip) keeps its own layout; these
// launches are the op-by-op form a VM program dispatches.
#include "si_internal.hpp"
#include "si_transformer.hpp"
#include "si_lanes.hpp"

#include <hip/hip_fp16.h>

namespace si {
namespace {

constexpr int NORM_THREADS = 1024;

__device__ __forceinline__ float wave_sum_f(float v)
{
    for (int off = 32; off > 0; off >>= 1)
        v += __shfl_xor(v, off);
    return v;
}

// Sum over the workgroup (every thread gets it); `red` holds one float per wave.
template <int THREADS>
__device__ __forceinline__ float block_sum(float v, float* red)
{
    v = wave_sum_f(v);
    if ((threadIdx.x & 63) == 0)
        red[threadIdx.x >> 6] = v;
    __syncthreads();
    float t = 0.0f;
#pragma unroll
    for (int w = 0; w < THREADS / 64; w++)
        t += red[w];
    __syncthreads();
    return t;
}

// One workgroup: the sum of squares of (hidden [+ residual]) over n values,
// then out_j = v_j * scale * w_j (the reference's operation order).
template <bool RESIDUAL>
__global__ __launch_bounds__(NORM_THREADS) void rms_norm_kernel(const float* __restrict__ hidden,
                                                                const float* __restrict__ residual,
                                                                const float* __restrict__ weight,
                                                                float* __restrict__ updated, float* __restrict__ out,
                                                                int n, float eps)
{
    __shared__ float red[NORM_THREADS / 64];
    float ss = 0.0f;
    for (int j = threadIdx.x; j < n; j += NORM_THREADS) {
        float v = hidden[j];
        if (RESIDUAL) {
            v = v + residual[j];
            updated[j] = v;
        }
        ss = fmaf(v, v, ss);
    }
    const float total = block_sum<NORM_THREADS>(ss, red);
    const float scale = 1.0f / sqrtf(total / static_cast<float>(n) + eps);
    for (int j = threadIdx.x; j < n; j += NORM_THREADS) {
        // each thread re-reads only values it wrote itself above
        const float v = RESIDUAL ? updated[j] : hidden[j];
        out[j] = v * scale * weight[j];
    }
}

__global__ __launch_bounds__(256) void swiglu_kernel(const float* __restrict__ gate_up, float* __restrict__ out,
                                                     int64_t n)
{
    const int64_t i = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
    if (i < n) {
        const float g = gate_up[i];
        out[i] = g / (1.0f + expf(-g)) * gate_up[n + i];
    }
}

template <typename T>
__device__ __forceinline__ void store_cache(T* cache, int64_t i, float v);
template <>
__device__ __forceinline__ void store_cache<float>(float* cache, int64_t i, float v) { cache[i] = v; }
template <>
__device__ __forceinline__ void store_cache<__half>(__half* cache, int64_t i, float v) { cache[i] = __float2half_rn(v); }

// One thread per value of qkv = [q (query_size) | k (kv_size) | v (kv_size)].
template <typename T>
__global__ __launch_bounds__(256) void rope_kv_write_kernel(RopeKvWriteArgs a, T* __restrict__ kc, T* __restrict__ vc)
{
    const int total = a.query_size + 2 * a.kv_size;
    const int i = static_cast<int>(blockIdx.x) * 256 + threadIdx.x;
    const int token = *a.position;
    if (token < 0 || token >= a.context || i >= total)
        return;
    const int half = a.rotary_size / 2;
    auto rotate = [&](int local, float value) {
        const int d = local % a.head_size;
        if (d >= a.rotary_size)
            return value;
        const int ri = d < half ? d : d - half;
        const int pair = d < half ? i + half : i - half;
        const float angle = static_cast<float>(token) * a.frequencies[ri];
        const float c = cosf(angle) * a.rope_scale, s = sinf(angle) * a.rope_scale;
        const float other = a.qkv[pair];
        return d < half ? value * c - other * s : value * c + other * s;
    };
    const float value = a.qkv[i];
    if (i < a.query_size) {
        a.query[i] = rotate(i, value);
    } else if (i < a.query_size + a.kv_size) {
        const int local = i - a.query_size;
        store_cache<T>(kc, static_cast<int64_t>(token) * a.kv_size + local, rotate(local, value));
    } else {
        const int local = i - a.query_size - a.kv_size;
        store_cache<T>(vc, static_cast<int64_t>(token) * a.kv_size + local, value);
    }
}

// 8 consecutive floats (two 16-byte loads).
__device__ __forceinline__ void load8(const float* p, float* f)
{
    const float4 a = reinterpret_cast<const float4*>(p)[0], b = reinterpret_cast<const float4*>(p)[1];
    f[0] = a.x; f[1] = a.y; f[2] = a.z; f[3] = a.w;
    f[4] = b.x; f[5] = b.y; f[6] = b.z; f[7] = b.w;
}

constexpr int GQA_THREADS = 256;
constexpr int GQA_CHUNK = 64;      // cache rows per partial of the workspace layout

// One workgroup = one KV head x CHUNK cache rows x up to G query heads of its
// group (grid z: the group in parts of at most 4 heads), every intermediate
// in registers (the decode step's form, without its rotary and append:
// rope-kv-write has already rotated the query and written the row).
// A cache row's HEAD values are SL = HEAD / 8 slices of 8; thread (wave w,
// lane l) takes slice l % SL of rows w * CHUNK / 4 + l / SL + RPW j for both
// the scores and the values, so the softmax weights stay in its registers.
// Every K and V row of the chunk is requested at once; each wave keeps its
// own maximum, and the waves' rows merge (with rescaling) through LDS at the
// kernel's one barrier.  Rows past the active range count as absent.
// Partials (m, l, o) of each query head and chunk go to the workspace at the
// 64-row layout's index (chunk < its chunk count).
//
// Bound: the round trips position -> cache rows -> partials (two launches a
// call), not the cache bytes.  FP32 caches, 32 heads of 64 over 4 KV heads,
// 4000 of 4096 rows, eight calls in a plan: 392 us with the staged form this
// replaces (scores and weights through LDS, one workgroup per query head,
// so a group's cache rows were read once per query head, and a merge that
// walked the chunks one by one on 32 workgroups of one wave: 17 + 31 us a
// call), 8.5 us a call now; 8 heads-of-128 groups of 4, fp16, 16000 of 16384
// rows: 59.4 -> 22.2 us; 512-row FP32 cache, 8 heads over 4: 7.7 -> 5.9 us.
template <typename T>
struct CacheSlice {   // 8 consecutive values of one cache row as loaded
    uint4 w[sizeof(T) == 2 ? 1 : 2];
};
template <typename T>
__device__ __forceinline__ CacheSlice<T> load_slice(const T* p)
{
    CacheSlice<T> r;
#pragma unroll
    for (int i = 0; i < (sizeof(T) == 2 ? 1 : 2); i++)
        r.w[i] = reinterpret_cast<const uint4*>(p)[i];
    return r;
}
__device__ __forceinline__ void unpack_slice(const CacheSlice<__half>& r, float* f)
{
    const uint32_t w[4] = {r.w[0].x, r.w[0].y, r.w[0].z, r.w[0].w};
#pragma unroll
    for (int k = 0; k < 4; k++) {
        f[2 * k] = __half2float(__ushort_as_half(static_cast<unsigned short>(w[k] & 0xffffu)));
        f[2 * k + 1] = __half2float(__ushort_as_half(static_cast<unsigned short>(w[k] >> 16)));
    }
}
__device__ __forceinline__ void unpack_slice(const CacheSlice<float>& r, float* f)
{
    f[0] = __uint_as_float(r.w[0].x); f[1] = __uint_as_float(r.w[0].y);
    f[2] = __uint_as_float(r.w[0].z); f[3] = __uint_as_float(r.w[0].w);
    f[4] = __uint_as_float(r.w[1].x); f[5] = __uint_as_float(r.w[1].y);
    f[6] = __uint_as_float(r.w[1].z); f[7] = __uint_as_float(r.w[1].w);
}

// Sum over the SL (8, 16 or 32) lanes that hold one cache row.
template <int SL>
__device__ __forceinline__ float slice_sum(float v)
{
    v = row_sum<SL < 16 ? SL : 16>(v);
    if constexpr (SL == 32) {
        const auto b = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
        v = __uint_as_float(b[0]) + __uint_as_float(b[1]);
    }
    return v;
}

// Maximum over the wave of values that are equal within a row's SL lanes.
template <int SL>
__device__ __forceinline__ float slices_max(float v)
{
    if constexpr (SL == 8)
        v = fmaxf(v, dpp_row<0x128>(v));   // the other row of the 16 lanes
    return rows_max(v);
}

template <typename T, int HEAD, int G, int CHUNK>
__global__ __launch_bounds__(GQA_THREADS) void gqa_chunk_kernel(GqaArgs a, const T* __restrict__ kc,
                                                                const T* __restrict__ vc)
{
    constexpr int SL = HEAD / 8, RPW = 64 / SL;        // lanes per cache row, rows per wave and step
    constexpr int WROWS = CHUNK / 4, PPL = WROWS / RPW;   // rows per wave, per lane
    static_assert(PPL * RPW * 4 == CHUNK, "whole rows per lane");
    const int g = blockIdx.x, chunk = blockIdx.y;
    const int group = a.query_heads / a.kv_heads;
    const int h0 = static_cast<int>(blockIdx.z) * G;   // first head of this part of the group
    const int start = chunk * CHUNK;
    const int t = threadIdx.x, lane = t & 63;
    const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
    const int dg = lane & (SL - 1), row = lane / SL;
    float q[G][8];
#pragma unroll
    for (int h = 0; h < G; h++)   // a last part with fewer heads repeats the group's last one and drops it
        load8(a.query + static_cast<int64_t>(g * group + min(h0 + h, group - 1)) * HEAD + 8 * dg, q[h]);
    const int active = min(max(*a.position, 0), a.context - 1);
    const bool valid = start <= active;
    const int count = min(CHUNK, active + 1 - start);
    const int64_t row_stride = static_cast<int64_t>(a.kv_heads) * HEAD;
    const T* kb = kc + static_cast<int64_t>(g) * HEAD + 8 * dg;
    const T* vb = vc + static_cast<int64_t>(g) * HEAD + 8 * dg;
    CacheSlice<T> kr[PPL], vr[PPL];
    if (valid) {   // a chunk past the active rows loads nothing and stores nothing
#pragma unroll
        for (int j = 0; j < PPL; j++) {
            const int64_t r = min(start + wave * WROWS + row + RPW * j, a.context - 1);
            kr[j] = load_slice(kb + r * row_stride);
            vr[j] = load_slice(vb + r * row_stride);
        }
    }
    // scores q.k / sqrt(HEAD), masked past the count; exponentials with the
    // hardware exp2 (__expf: L2 error against 64 bits as with expf to two
    // digits, for scores of standard deviation 1, 4 and 16; expf costs 6 to 15%)
    const float rscale = 1.0f / sqrtf(static_cast<float>(HEAD));
    float sc[G][PPL];
#pragma unroll
    for (int j = 0; j < PPL; j++) {
        const int p = wave * WROWS + row + RPW * j;
        float k8[8];
        unpack_slice(kr[j], k8);
#pragma unroll
        for (int h = 0; h < G; h++) {
            float d = 0.0f;
#pragma unroll
            for (int e = 0; e < 8; e++)
                d = fmaf(q[h][e], k8[e], d);
            d = slice_sum<SL>(d);
            sc[h][j] = p < count ? d * rscale : -INFINITY;
        }
    }
    float m[G], l[G], acc[G][8];
#pragma unroll
    for (int h = 0; h < G; h++) {
        float mh = sc[h][0];
#pragma unroll
        for (int j = 1; j < PPL; j++)
            mh = fmaxf(mh, sc[h][j]);
        mh = slices_max<SL>(mh);
        m[h] = mh;
        float lh = 0.0f;
#pragma unroll
        for (int j = 0; j < PPL; j++) {
            const float e = sc[h][j] == -INFINITY ? 0.0f : __expf(sc[h][j] - mh);
            sc[h][j] = e;
            lh += e;
        }
        l[h] = lh;
#pragma unroll
        for (int e = 0; e < 8; e++)
            acc[h][e] = 0.0f;
    }
#pragma unroll
    for (int j = 0; j < PPL; j++) {
        const int p = wave * WROWS + row + RPW * j;
        float v8[8];
        unpack_slice(vr[j], v8);
#pragma unroll
        for (int e = 0; e < 8; e++)
            v8[e] = p < count ? v8[e] : 0.0f;   // rows past the count may hold anything
#pragma unroll
        for (int h = 0; h < G; h++)
#pragma unroll
            for (int e = 0; e < 8; e++)
                acc[h][e] = fmaf(sc[h][j], v8[e], acc[h][e]);
    }
    __shared__ float4 red4[4 * RPW][G][HEAD / 4];
    __shared__ float wm[4][G], wl[4 * RPW][G];
#pragma unroll
    for (int h = 0; h < G; h++) {
        red4[wave * RPW + row][h][2 * dg] = make_float4(acc[h][0], acc[h][1], acc[h][2], acc[h][3]);
        red4[wave * RPW + row][h][2 * dg + 1] = make_float4(acc[h][4], acc[h][5], acc[h][6], acc[h][7]);
    }
    if (dg == 0)
#pragma unroll
        for (int h = 0; h < G; h++) {
            wl[wave * RPW + row][h] = l[h];
            if (row == 0)
                wm[wave][h] = m[h];
        }
    __syncthreads();
    if (!valid)
        return;
    const float* red = reinterpret_cast<const float*>(red4);
    for (int i = t; i < G * HEAD; i += GQA_THREADS) {
        const int h = i / HEAD, d = i % HEAD;
        if (h0 + h >= group)
            break;
        const float M = fmaxf(fmaxf(wm[0][h], wm[1][h]), fmaxf(wm[2][h], wm[3][h]));   // finite: row start is active
        float o = 0.0f, lsum = 0.0f;
#pragma unroll
        for (int w = 0; w < 4; w++) {
            const float f = wm[w][h] == -INFINITY ? 0.0f : __expf(wm[w][h] - M);   // a wave without active rows adds nothing
            float ow = 0.0f, lw = 0.0f;
#pragma unroll
            for (int r = 0; r < RPW; r++) {
                ow += red[((w * RPW + r) * G + h) * HEAD + d];
                lw += wl[w * RPW + r][h];
            }
            o = fmaf(ow, f, o);
            lsum = fmaf(lw, f, lsum);
        }
        if (gridDim.y == 1) {   // the cache is one chunk: no merge follows
            a.output[static_cast<int64_t>(g * group + h0 + h) * HEAD + d] = o / lsum;
            continue;
        }
        float* dst = a.workspace + (static_cast<int64_t>(g * group + h0 + h) * a.chunks + chunk) * (HEAD + 2);
        dst[2 + d] = o;
        if (d == 0) {
            dst[0] = M;
            dst[1] = lsum;
        }
    }
}

// The merge of CHUNK-row partials, one workgroup per query head:
// out = sum_c o_c e^(m_c - M) / sum_c l_c e^(m_c - M) over the active
// chunks, M = max_c m_c.  SLOTS groups of HEAD threads take the chunks in
// turn, each a batch of BATCH chunks per round trip merged online (m, l, o
// rescaled per batch), and merge through LDS: up to BATCH * SLOTS chunks
// cost one round trip, the first batch's requested before the position is
// known.  Lane u (mod BATCH) holds (m, l) of the batch's chunk u, so a wave
// issues BATCH + 2 loads for it and not 3 BATCH: 48 loads of 16 waves held the
// address unit for longer than the merge of a few chunks needs (168 of 2800
// rows, 6 heads of 128 over 2: 9.4 us a call, 7.5 now; 16383 of 16384, 16 over
// 4: 17.4, 15.8 now).
template <int HEAD, int CHUNK, int SLOTS, int BATCH>
__global__ __launch_bounds__(HEAD * SLOTS) void gqa_merge_kernel(GqaArgs a)
{
    static_assert(HEAD % 64 == 0 && BATCH <= 16, "a slot is whole waves, a batch's (m, l) one row of lanes");
    const int head = blockIdx.x, d = threadIdx.x % HEAD, own = threadIdx.x % BATCH;
    const int slot = __builtin_amdgcn_readfirstlane(threadIdx.x / HEAD);
    const float* src = a.workspace + static_cast<int64_t>(head) * a.chunks * (HEAD + 2);
    const int all = (a.context + CHUNK - 1) / CHUNK;   // partials a full cache has
    const int active = min(max(*a.position, 0), a.context - 1);
    const int n = active / CHUNK + 1;
    float m = -INFINITY, L = 0.0f, O = 0.0f;
    int c0 = slot;
    do {   // the first batch's loads (any partial of the workspace) need no position
        const float* pc = src + static_cast<int64_t>(min(c0 + own * SLOTS, all - 1)) * (HEAD + 2);
        const float mc = pc[0], lc = pc[1];
        float oc[BATCH];
#pragma unroll
        for (int u = 0; u < BATCH; u++)
            oc[u] = src[static_cast<int64_t>(min(c0 + u * SLOTS, all - 1)) * (HEAD + 2) + 2 + d];
        const bool in = c0 + own * SLOTS < n;   // partials past the active chunks may hold anything
        const float bm = fmaxf(m, row_max<BATCH>(in ? mc : -INFINITY));
        const float r = m == -INFINITY ? 0.0f : __expf(m - bm);
        const float e = in ? __expf(mc - bm) : 0.0f;
        L = fmaf(L, r, row_sum<BATCH>(in ? lc * e : 0.0f));
        O *= r;
#pragma unroll
        for (int u = 0; u < BATCH; u++) {
            const float eu = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(e), u));
            O = fmaf(c0 + u * SLOTS < n ? oc[u] : 0.0f, eu, O);
        }
        m = bm;
        c0 += BATCH * SLOTS;
    } while (c0 < n);
    __shared__ float sm[SLOTS], sl[SLOTS], so[SLOTS][HEAD];
    so[slot][d] = O;
    if (d == 0) {
        sm[slot] = m;
        sl[slot] = L;
    }
    __syncthreads();
    if (slot != 0)
        return;
    float M = sm[0];
#pragma unroll
    for (int s = 1; s < SLOTS; s++)
        M = fmaxf(M, sm[s]);
    float lsum = 0.0f, o = 0.0f;
#pragma unroll
    for (int s = 0; s < SLOTS; s++) {
        const float e = __expf(sm[s] - M);   // a slot without chunks: m = -inf, e = 0
        lsum = fmaf(sl[s], e, lsum);
        o = fmaf(so[s][d], e, o);
    }
    a.output[static_cast<int64_t>(head) * HEAD + d] = o / lsum;
}

template <typename T, int HEAD, int G, int CHUNK>
hipError_t launch_gqa_form(const GqaArgs& a, int parts, hipStream_t s)
{
    const int chunks = (a.context + CHUNK - 1) / CHUNK;
    const dim3 grid(static_cast<unsigned>(a.kv_heads), static_cast<unsigned>(chunks), static_cast<unsigned>(parts));
    hipLaunchKernelGGL((gqa_chunk_kernel<T, HEAD, G, CHUNK>), grid, dim3(GQA_THREADS), 0, s, a,
                       static_cast<const T*>(a.key_cache), static_cast<const T*>(a.value_cache));
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess || chunks == 1)
        return e;
    // no more slots and loads than one round trip for every chunk takes, up to
    // 128 chunks (64 at 256-value heads); the 256 chunks of 16384 rows over one
    // KV head take two (four)
    const dim3 heads(static_cast<unsigned>(a.query_heads));
    if (chunks <= 8)
        hipLaunchKernelGGL((gqa_merge_kernel<HEAD, CHUNK, 1, 8>), heads, dim3(HEAD), 0, s, a);
    else if (chunks <= 32)
        hipLaunchKernelGGL((gqa_merge_kernel<HEAD, CHUNK, 4, 8>), heads, dim3(HEAD * 4), 0, s, a);
    else {
        constexpr int SLOTS = HEAD == 256 ? 4 : 8;
        hipLaunchKernelGGL((gqa_merge_kernel<HEAD, CHUNK, SLOTS, 16>), heads, dim3(HEAD * SLOTS), 0, s, a);
    }
    return hipGetLastError();
}

// CHUNK: 128 rows where the whole cache then still gives a workgroup per CU
// (half the partials to merge), 64 otherwise (2000-row cache, 8 KV heads of
// 128: 8.8 us against 10.0 with 128 rows; 1 KV head, 16384 rows of 128 in
// FP32: 13.2 against 15.9 with 128 rows only from 512 workgroups); 256-value
// heads keep 64 (a lane's rows of a 128-row chunk would not fit its
// registers).  A cache of at most 128 rows is one chunk and needs no merge.
template <typename T, int HEAD, int G>
hipError_t launch_gqa_group(const GqaArgs& a, int parts, hipStream_t s)
{
    if constexpr (HEAD < 256) {
        if (a.context <= 128 || static_cast<int64_t>(a.kv_heads) * parts * ((a.context + 127) / 128) >= 256)
            return launch_gqa_form<T, HEAD, G, 128>(a, parts, s);
    }
    return launch_gqa_form<T, HEAD, G, 64>(a, parts, s);
}

template <typename T, int HEAD>
hipError_t launch_gqa_head(const GqaArgs& a, hipStream_t s)
{
    const int group = a.query_heads / a.kv_heads;
    const int parts = (group + 3) / 4;
    switch ((group + parts - 1) / parts) {   // heads per part, evenly
    case 1: return launch_gqa_group<T, HEAD, 1>(a, parts, s);
    case 2: return launch_gqa_group<T, HEAD, 2>(a, parts, s);
    case 3: return launch_gqa_group<T, HEAD, 3>(a, parts, s);
    default: return launch_gqa_group<T, HEAD, 4>(a, parts, s);
    }
}

}  // namespace

hipError_t launch_rms_norm(const float* x, const float* w, float* out, int n, float eps, hipStream_t s)
{
    hipLaunchKernelGGL((rms_norm_kernel<false>), dim3(1), dim3(NORM_THREADS), 0, s, x, nullptr, w, nullptr, out, n, eps);
    return hipGetLastError();
}

hipError_t launch_residual_rms_norm(const float* hidden, const float* residual, const float* w, float* updated,
                                    float* out, int n, float eps, hipStream_t s)
{
    hipLaunchKernelGGL((rms_norm_kernel<true>), dim3(1), dim3(NORM_THREADS), 0, s, hidden, residual, w, updated, out, n,
                       eps);
    return hipGetLastError();
}

hipError_t launch_swiglu(const float* gate_up, float* out, int64_t n, hipStream_t s)
{
    hipLaunchKernelGGL(swiglu_kernel, dim3(static_cast<unsigned>((n + 255) / 256)), dim3(256), 0, s, gate_up, out, n);
    return hipGetLastError();
}

hipError_t launch_rope_kv_write(const RopeKvWriteArgs& a, hipStream_t s)
{
    const int total = a.query_size + 2 * a.kv_size;
    const dim3 grid(static_cast<unsigned>((total + 255) / 256));
    if (a.cache_fp16)
        hipLaunchKernelGGL((rope_kv_write_kernel<__half>), grid, dim3(256), 0, s, a, static_cast<__half*>(a.key_cache),
                           static_cast<__half*>(a.value_cache));
    else
        hipLaunchKernelGGL((rope_kv_write_kernel<float>), grid, dim3(256), 0, s, a, static_cast<float*>(a.key_cache),
                           static_cast<float*>(a.value_cache));
    return hipGetLastError();
}

int64_t gqa_workspace_floats(int query_heads, int head_size, int context)
{
    return static_cast<int64_t>(query_heads) * ((context + GQA_CHUNK - 1) / GQA_CHUNK) * (head_size + 2);
}

hipError_t launch_gqa(const GqaArgs& a, hipStream_t s)
{
    if (a.kv_heads < 1 || a.query_heads < 1 || a.query_heads % a.kv_heads != 0)
        return hipErrorInvalidValue;
    switch (a.head_size) {
    case 64: return a.cache_fp16 ? launch_gqa_head<__half, 64>(a, s) : launch_gqa_head<float, 64>(a, s);
    case 128: return a.cache_fp16 ? launch_gqa_head<__half, 128>(a, s) : launch_gqa_head<float, 128>(a, s);
    case 256: return a.cache_fp16 ? launch_gqa_head<__half, 256>(a, s) : launch_gqa_head<float, 256>(a, s);
    default: return hipErrorInvalidValue;
    }
}

}  // namespace si
