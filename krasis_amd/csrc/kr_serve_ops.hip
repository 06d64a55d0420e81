// kr_serve_ops.hip -- row kernels of the batched serving step (gfx950, wave64): embedding, layer / RMS norm, rotary table, query / key preparation with
// the paged cache append, sliding-window attention with a sink over the paged cache, group-limited top-k router, expert row sort, gated activations,
// the parallel-block residual sum, argmax.
//
// Every f32 reduction here is a lane / wave tree; sums written as a * b + c may be contracted (explicit __builtin_fmaf): the serving path states a
// tolerance against an f32 restatement, not a bit pattern.
#include <hip/hip_runtime.h>
#include <limits.h>
#include <math.h>
#include <stdint.h>

#include <algorithm>
#include <initializer_list>
#include <type_traits>

#include "kr_device.h"
#include "kr_lds_optin.h"
#include "kr_serve_gemm_dev.h"
#include "kr_serve_ops.h"

namespace {
__device__ __forceinline__ float sv_ld(const float* p) { return *p; }
__device__ __forceinline__ float sv_ld(const uint16_t* p) { return kr_bf16_to_f32(*p); }
__device__ __forceinline__ void sv_st(float* p, float v) { *p = v; }
__device__ __forceinline__ void sv_st(uint16_t* p, float v) { *p = kr_f32_to_bf16(v); }

// wave-wide sum / maximum, every lane receives it: four DPP steps inside each row of 16 lanes, then the four rows through scalar reads
#define SV_DPPF(v, ctrl) __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), (ctrl), 0xF, 0xF, false))
#define SV_LANE(v, i) __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), (i)))
__device__ __forceinline__ float sv_wave_sum(float v) {
    v += SV_DPPF(v, KR_DPP_XOR1); v += SV_DPPF(v, KR_DPP_XOR2); v += SV_DPPF(v, KR_DPP_HALF_MIRROR); v += SV_DPPF(v, KR_DPP_MIRROR);
    return (SV_LANE(v, 0) + SV_LANE(v, 16)) + (SV_LANE(v, 32) + SV_LANE(v, 48));
}
__device__ __forceinline__ float sv_wave_max(float v) {
    v = fmaxf(v, SV_DPPF(v, KR_DPP_XOR1)); v = fmaxf(v, SV_DPPF(v, KR_DPP_XOR2)); v = fmaxf(v, SV_DPPF(v, KR_DPP_HALF_MIRROR)); v = fmaxf(v, SV_DPPF(v, KR_DPP_MIRROR));
    return fmaxf(fmaxf(SV_LANE(v, 0), SV_LANE(v, 16)), fmaxf(SV_LANE(v, 32), SV_LANE(v, 48)));
}
// sum over a workgroup of NW waves; every thread receives it
template <int NW>
__device__ __forceinline__ float sv_block_sum(float v, float* red) {
    v = sv_wave_sum(v);
    if constexpr (NW == 1) return v;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    __syncthreads();
    if (lane == 0) red[wave] = v;
    __syncthreads();
    float s = 0.0f;
#pragma unroll
    for (int w = 0; w < NW; w++) s += red[w];
    return s;
}

template <typename T>
__global__ void __launch_bounds__(256) sv_embed_kernel(const T* __restrict__ table, const int* __restrict__ tokens, float* __restrict__ x, T* __restrict__ h_out, int width,
                                                       float scale, const T* __restrict__ table2, const int* __restrict__ rows2) {
    const int t = blockIdx.x;
    const T* row = table + (size_t)tokens[t] * width;
    const T* row2 = table2 ? table2 + (size_t)rows2[t] * width : nullptr;
    for (int c = threadIdx.x; c < width; c += 256) {
        float v = sv_ld(row + c) * scale;
        if (row2) v += sv_ld(row2 + c);
        x[(size_t)t * width + c] = v;
        if (h_out) sv_st(h_out + (size_t)t * width + c, v);
    }
}

// statistics of `groups` equal consecutive parts of a row (LDS or global): st[2 g] = mean (0 for an RMS norm), st[2 g + 1] = 1 / sqrt(variance + eps).
// Wave w of the NW takes the parts w, w + NW, ...; the caller makes the row visible before and synchronises after.
template <int KIND, int NW = 4>
__device__ __forceinline__ void sv_group_stats(const float* xr, int width, int groups, float eps, float* st) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, gw = width / groups;
    for (int g = wave; g < groups; g += NW) {
        const float* xg = xr + (size_t)g * gw;
        float mean = 0.0f;
        if constexpr (KIND == KR_SV_NORM_LAYER) {
            float s = 0.0f;
            for (int c = lane; c < gw; c += 64) s += xg[c];
            mean = sv_wave_sum(s) / (float)gw;
        }
        float q = 0.0f;
        for (int c = lane; c < gw; c += 64) { const float d = xg[c] - mean; q = __builtin_fmaf(d, d, q); }
        q = sv_wave_sum(q);
        if (lane == 0) { st[2 * g] = mean; st[2 * g + 1] = 1.0f / sqrtf(q / (float)gw + eps); }
    }
}

template <typename T, int KIND>
__global__ void __launch_bounds__(256) sv_norm_kernel(const float* __restrict__ x, const int* __restrict__ rows, const float* __restrict__ w, const float* __restrict__ b,
                                                      T* __restrict__ out, int width, float eps, int groups, float* __restrict__ out32) {
    __shared__ float red[4];
    extern __shared__ float gst[];            // [2 * groups] when the row is normed in parts
    const int r = blockIdx.x;
    const float* xr = x + (size_t)(rows ? rows[r] : r) * width;
    if (groups > 1) {
        sv_group_stats<KIND>(xr, width, groups, eps, gst);
        __syncthreads();
        const int gw = width / groups;
        for (int c = threadIdx.x; c < width; c += 256) {
            const int g = c / gw;
            float v = (xr[c] - gst[2 * g]) * gst[2 * g + 1] * w[c];
            if (b) v += b[c];
            sv_st(out + (size_t)r * width + c, v);
            if (out32) out32[(size_t)r * width + c] = v;
        }
        return;
    }
    float mean = 0.0f;
    if constexpr (KIND == KR_SV_NORM_LAYER) {
        float s = 0.0f;
        for (int c = threadIdx.x; c < width; c += 256) s += xr[c];
        mean = sv_block_sum<4>(s, red) / (float)width;
    }
    float q = 0.0f;
    for (int c = threadIdx.x; c < width; c += 256) { const float d = xr[c] - mean; q = __builtin_fmaf(d, d, q); }
    const float var = sv_block_sum<4>(q, red) / (float)width;
    const float inv = 1.0f / sqrtf(var + eps);
    for (int c = threadIdx.x; c < width; c += 256) {
        float v = (xr[c] - mean) * inv * w[c];
        if (b) v += b[c];
        sv_st(out + (size_t)r * width + c, v);
        if (out32) out32[(size_t)r * width + c] = v;
    }
}

// ---- the same rows four columns at a time, a row held in its workgroup's registers (thread: columns 4 (tid + NT j), j < CH): read once, in 16-byte pieces that are all in flight
// together, and normed without a second pass over memory.  Bound by the latency of one round trip for a few rows and by the copy rate for many.  At 2048 columns, before (a scalar row
// kept in LDS) and after: residual of one row and six expert rows 8.6 -> 5.8 us, of 4096 such rows 115 -> 71 us; norm of one row 10 -> 3.3 us; embedding and norm 16.4 -> 4.0 us.
// Widths that are multiples of four up to 16 NT columns; other widths take the kernels around these.
__device__ __forceinline__ float4 sv_ld4(const float* p) { return *reinterpret_cast<const float4*>(p); }
__device__ __forceinline__ float4 sv_ld4(const uint16_t* p) {
    const uint2 u = *reinterpret_cast<const uint2*>(p);
    return make_float4(__uint_as_float(u.x << 16), __uint_as_float(u.x & 0xFFFF0000u), __uint_as_float(u.y << 16), __uint_as_float(u.y & 0xFFFF0000u));
}
__device__ __forceinline__ void sv_st4(float* p, float4 v) { *reinterpret_cast<float4*>(p) = v; }
__device__ __forceinline__ void sv_st4(uint16_t* p, float4 v) {
    *reinterpret_cast<uint2*>(p) = make_uint2(kr_f32_to_bf16(v.x) | ((uint32_t)kr_f32_to_bf16(v.y) << 16), kr_f32_to_bf16(v.z) | ((uint32_t)kr_f32_to_bf16(v.w) << 16));
}
// v <- (v - mean) / sqrt(variance + eps) * w (+ b) over the row; groups > 1: every part of the row by its own statistics (row: LDS [width] | [2 groups])
template <int KIND, int NT, int CH>
__device__ __forceinline__ void sv_row_norm(float4 (&v)[CH], int width, int groups, float eps, const float* w, const float* b, float* red, float* row) {
    float mean = 0.0f, inv = 0.0f;
    float* gst = row + width;
    if (groups > 1) {
        __syncthreads();
#pragma unroll
        for (int j = 0; j < CH; j++) { const int c = 4 * (threadIdx.x + NT * j); if (c < width) sv_st4(row + c, v[j]); }
        __syncthreads();
        sv_group_stats<KIND, NT / 64>(row, width, groups, eps, gst);
        __syncthreads();
    } else {
        if constexpr (KIND == KR_SV_NORM_LAYER) {
            float s = 0.0f;
#pragma unroll
            for (int j = 0; j < CH; j++) if (4 * (threadIdx.x + NT * j) < width) s += (v[j].x + v[j].y) + (v[j].z + v[j].w);
            mean = sv_block_sum<NT / 64>(s, red) / (float)width;
        }
        float q = 0.0f;
#pragma unroll
        for (int j = 0; j < CH; j++) {
            if (4 * (threadIdx.x + NT * j) >= width) continue;
            const float dx = v[j].x - mean, dy = v[j].y - mean, dz = v[j].z - mean, dw = v[j].w - mean;
            q = __builtin_fmaf(dx, dx, q); q = __builtin_fmaf(dy, dy, q); q = __builtin_fmaf(dz, dz, q); q = __builtin_fmaf(dw, dw, q);
        }
        inv = 1.0f / sqrtf(sv_block_sum<NT / 64>(q, red) / (float)width + eps);
    }
    const int gw = groups > 1 ? width / groups : width;
#pragma unroll
    for (int j = 0; j < CH; j++) {
        const int c = 4 * (threadIdx.x + NT * j);
        if (c >= width) continue;
        const float4 ww = sv_ld4(w + c), bb = b ? sv_ld4(b + c) : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
        float m[4] = {mean, mean, mean, mean}, r[4] = {inv, inv, inv, inv};
        if (groups > 1) {
#pragma unroll
            for (int e = 0; e < 4; e++) { m[e] = gst[2 * ((c + e) / gw)]; r[e] = gst[2 * ((c + e) / gw) + 1]; }
        }
        v[j] = make_float4((v[j].x - m[0]) * r[0] * ww.x + bb.x, (v[j].y - m[1]) * r[1] * ww.y + bb.y, (v[j].z - m[2]) * r[2] * ww.z + bb.z, (v[j].w - m[3]) * r[3] * ww.w + bb.w);
    }
}
template <typename T, int KIND, int NT, int CH>
__global__ void __launch_bounds__(NT) sv_norm_vec_kernel(const float* __restrict__ x, const int* __restrict__ rows, const float* __restrict__ w, const float* __restrict__ b,
                                                         T* __restrict__ out, int width, float eps, int groups, float* __restrict__ out32) {
    __shared__ float red[NT / 64];
    extern __shared__ __attribute__((aligned(16))) float row[];
    const size_t r = blockIdx.x;
    const float* xr = x + (size_t)(rows ? rows[r] : r) * width;
    float4 v[CH];
#pragma unroll
    for (int j = 0; j < CH; j++) { const int c = 4 * (threadIdx.x + NT * j); if (c < width) v[j] = sv_ld4(xr + c); }
    sv_row_norm<KIND, NT, CH>(v, width, groups, eps, w, b, red, row);
#pragma unroll
    for (int j = 0; j < CH; j++) {
        const int c = 4 * (threadIdx.x + NT * j);
        if (c < width) { sv_st4(out + r * width + c, v[j]); if (out32) sv_st4(out32 + r * width + c, v[j]); }
    }
}
// cos / sin of one (token, frequency)
__device__ __forceinline__ float2 sv_rope_angle(int pos, double inv_freq, float mult) {
    const double a = (double)pos * inv_freq;
    return make_float2((float)cos(a) * mult, (float)sin(a) * mult);
}
__global__ void sv_rope_table_kernel(const int* __restrict__ pos, const double* __restrict__ inv_freq, float2* __restrict__ cs, int T, int half, float mult) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= T * half) return;
    const int t = i / half, j = i - t * half;
    cs[i] = sv_rope_angle(pos[t], inv_freq[j], mult);
}

// what a step's arrays need before its first layer, straight from the pinned host memory they were written to: the copy that later launches read, and the rotation tables.
// A copy command, the tables and the embedding were three launches in a row of 4 - 5 us each; none needs another's result.
// Every lane's read of host memory is a request of its own over the link (twelve requests' arrays word by word: 18 us), so the copy takes 16 bytes a lane and a position is
// read once per workgroup.  System scope: host memory must not come from a cache line of the step before.
__device__ __forceinline__ int sv_host_word(const int* p) { return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM); }
__device__ __forceinline__ int sv_host_word_wave(const int* p) {      // one address per wave
    int v = 0;
    if ((threadIdx.x & 63) == 0) v = sv_host_word(p);
    return __builtin_amdgcn_readfirstlane(v);
}
__device__ __forceinline__ void sv_begin(const KrSvBegin& b, const int block, const int blocks, const int nt) {
    __shared__ int pos[64];
    const int n = blocks * nt, i0 = block * nt + threadIdx.x;
    if ((int)threadIdx.x < b.T) pos[threadIdx.x] = sv_host_word(b.src + b.pos_at + threadIdx.x);      // (T <= 64)
    for (int i = i0; i < (b.words + 3) / 4; i += n) {
        gu4 v;
        asm volatile("global_load_dwordx4 %0, %1, off sc0 sc1\n\ts_waitcnt vmcnt(0)" : "=&v"(v) : "v"(b.src + 4 * i) : "memory");
        *reinterpret_cast<gu4*>(b.dst + 4 * i) = v;
    }
    __syncthreads();
    for (int i = i0; i < b.T * b.halves; i += n) {
        int j = i;
        for (int r = 0; r < b.n_rope; r++) {
            const int m = b.T * b.rope[r].half;
            if (j < m) { b.rope[r].cs[j] = sv_rope_angle(pos[j / b.rope[r].half], b.rope[r].inv_freq[j % b.rope[r].half], b.rope[r].mult); break; }
            j -= m;
        }
    }
}
__global__ void __launch_bounds__(256) sv_begin_kernel(const KrSvBegin b) { sv_begin(b, blockIdx.x, gridDim.x, 256); }
static int sv_begin_blocks(const KrSvBegin& b, int nt) { return std::max(1, std::min(64, std::max((b.words + 3) / 4, b.T * b.halves) / nt + 1)); }

// the token's row (scaled, a second table's row added), to the stream and, normed, to the first sublayer
template <typename T, int KIND, int NT, int CH>
__global__ void __launch_bounds__(NT) sv_embed_norm_kernel(const T* __restrict__ table, const int* __restrict__ tokens, float* __restrict__ x, float scale, const T* __restrict__ table2,
                                                           const int* __restrict__ rows2, const float* __restrict__ w, const float* __restrict__ b, T* __restrict__ out, int width, float eps,
                                                           int groups, float* __restrict__ out32, const KrSvBegin bg, const int R) {
    __shared__ float red[NT / 64];
    extern __shared__ __attribute__((aligned(16))) float row[];
    const size_t t = blockIdx.x;
    if ((int)t >= R) { sv_begin(bg, (int)t - R, gridDim.x - R, NT); return; }      // (bg.words > 0: tokens and rows2 are host memory)
    const T* e = table + (size_t)(bg.words > 0 ? sv_host_word_wave(tokens + t) : tokens[t]) * width;
    const T* e2 = table2 ? table2 + (size_t)(bg.words > 0 ? sv_host_word_wave(rows2 + t) : rows2[t]) * width : nullptr;
    float4 v[CH];
#pragma unroll
    for (int j = 0; j < CH; j++) {
        const int c = 4 * (threadIdx.x + NT * j);
        if (c >= width) continue;
        v[j] = sv_ld4(e + c);
        v[j] = make_float4(v[j].x * scale, v[j].y * scale, v[j].z * scale, v[j].w * scale);
        if (e2) { const float4 u = sv_ld4(e2 + c); v[j] = make_float4(v[j].x + u.x, v[j].y + u.y, v[j].z + u.z, v[j].w + u.w); }
        sv_st4(x + t * width + c, v[j]);
    }
    sv_row_norm<KIND, NT, CH>(v, width, groups, eps, w, b, red, row);
#pragma unroll
    for (int j = 0; j < CH; j++) {
        const int c = 4 * (threadIdx.x + NT * j);
        if (c < width) { sv_st4(out + t * width + c, v[j]); if (out32) sv_st4(out32 + t * width + c, v[j]); }
    }
}
// threads and chunks of a row kernel: decode-sized steps spread a row over many threads (its workgroup is alone on a compute unit and the chain is what the launch waits
// for), prompts take 256.  f(NT, CH) is the launch; false: the width is not for these kernels
template <typename F> static bool sv_vec_rows(int rows, int width, F f) {
    using std::integral_constant;
    if (width % 4 != 0 || width > 16384) return false;
    if (rows > 64 && width <= 1024) f(integral_constant<int, 256>{}, integral_constant<int, 1>{});
    else if (rows > 64 && width <= 2048) f(integral_constant<int, 256>{}, integral_constant<int, 2>{});
    else if (rows > 64 && width <= 4096) f(integral_constant<int, 256>{}, integral_constant<int, 4>{});
    else if (width <= 2048) f(integral_constant<int, 512>{}, integral_constant<int, 1>{});
    else if (width <= 4096) f(integral_constant<int, 1024>{}, integral_constant<int, 1>{});
    else f(integral_constant<int, 1024>{}, integral_constant<int, 4>{});
    return true;
}
// 16-byte pieces of every operand (a null pointer passes)
static bool sv_al16(std::initializer_list<const void*> ps) { for (const void* p : ps) if ((uintptr_t)p & 15) return false; return true; }

// input convolution over positions (KrSvCanon): one thread per (token, channel)
template <typename T>
__global__ void __launch_bounds__(256) sv_canon_kernel(const KrSvCanon a, T* __restrict__ out) {
    const int t = blockIdx.x, c = blockIdx.y * 256 + threadIdx.x;
    if (c >= a.width) return;
    const int p = a.pos[t], sl = a.slot[t], K = a.taps - 1;
    const float* w = a.w + (size_t)c * a.taps;
    float acc = a.h32[(size_t)t * a.width + c];
    acc = __builtin_fmaf(w[K], acc, acc);                     // the tap on the token itself
    for (int d = 1; d <= K; d++) {                            // d positions back
        const int q = p - d;
        if (q < 0) break;
        float hv;
        if (t - d >= 0 && a.slot[t - d] == sl) hv = a.h32[(size_t)(t - d) * a.width + c];
        else hv = a.state[((size_t)sl * K + q % K) * a.width + c];
        acc = __builtin_fmaf(w[K - d], hv, acc);
    }
    sv_st(out + (size_t)t * a.width + c, acc);
}

// the stream itself (kr_sv_stream_norm): a vector joins the row, and / or the row is normed -- in place, or into the next sublayer's input
template <typename T, int KIND>
__global__ void __launch_bounds__(256) sv_stream_norm_kernel(float* __restrict__ x, const float* __restrict__ add, const float* __restrict__ w, const float* __restrict__ b, int in_place,
                                                             T* __restrict__ out, int width, float eps, int groups) {
    extern __shared__ float xr[];            // [width] | [2 * groups]
    __shared__ float red[4];
    const size_t t = blockIdx.x;
    float* xp = x + t * width;
    float* gst = xr + width;
    float s1 = 0.0f;
    for (int c = threadIdx.x; c < width; c += 256) {
        float v = xp[c];
        if (add) { v += add[c]; xp[c] = v; }
        xr[c] = v; s1 += v;
    }
    if (!w) return;
    float mean = 0.0f, inv = 0.0f;
    if (groups > 1) { __syncthreads(); sv_group_stats<KIND, 4>(xr, width, groups, eps, gst); __syncthreads(); }
    else {
        if constexpr (KIND == KR_SV_NORM_LAYER) mean = sv_block_sum<4>(s1, red) / (float)width;
        float q = 0.0f;
        for (int c = threadIdx.x; c < width; c += 256) { const float dv = xr[c] - mean; q = __builtin_fmaf(dv, dv, q); }
        inv = 1.0f / sqrtf(sv_block_sum<4>(q, red) / (float)width + eps);
    }
    const int gw = groups > 1 ? width / groups : width;
    for (int c = threadIdx.x; c < width; c += 256) {
        if (groups > 1) { mean = gst[2 * (c / gw)]; inv = gst[2 * (c / gw) + 1]; }
        float v = (xr[c] - mean) * inv * w[c];
        if (b) v += b[c];
        if (in_place) xp[c] = v; else sv_st(out + t * width + c, v);
    }
}

// short convolution on the channels of a projection (KrSvChanConv): one thread per (token, channel)
__global__ void __launch_bounds__(256) sv_chan_conv_kernel(const KrSvChanConv a) {
    const int t = blockIdx.x, c = blockIdx.y * 256 + threadIdx.x;
    if (c >= a.C) return;
    const int p = a.pos[t], sl = a.slot[t], K = a.taps - 1;
    const float* w = a.w + (size_t)c * a.taps;
    const float ib = a.in_bias ? a.in_bias[c] : 0.0f;
    float acc = a.cb ? a.cb[c] : 0.0f;
    acc = __builtin_fmaf(w[K], a.in[(size_t)t * a.ld_in + c] + ib, acc);
    for (int d = 1; d <= K; d++) {            // d positions back
        const int q = p - d;
        if (q < 0) break;
        float u;
        if (t - d >= 0 && a.slot[t - d] == sl) u = a.in[(size_t)(t - d) * a.ld_in + c] + ib;
        else u = a.state[((size_t)sl * K + q % K) * a.C + c];
        acc = __builtin_fmaf(w[K - d], u, acc);
    }
    if (a.act == 1) acc = acc / (1.0f + expf(-acc));
    a.out[(size_t)t * a.ld_out + c] = acc;
}
// the last taps - 1 inputs of every portion -> the request's ring
__global__ void __launch_bounds__(256) sv_chan_conv_save_kernel(const KrSvChanConv a) {
    const int e = blockIdx.x, i = blockIdx.y, c = blockIdx.z * 256 + threadIdx.x, K = a.taps - 1;
    if (c >= a.C) return;
    const int t = a.ent_off[e + 1] - 1 - i;
    if (t < a.ent_off[e]) return;
    const float ib = a.in_bias ? a.in_bias[c] : 0.0f;
    a.state[((size_t)a.slot[t] * K + a.pos[t] % K) * a.C + c] = a.in[(size_t)t * a.ld_in + c] + ib;
}
__global__ void sv_scale_kernel(float* __restrict__ p, size_t n, float scale) {
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] *= scale;
}

// unit_norm == 3: 1 / rms over the whole q row (part 0) and the whole k row (part 1) of every token, biases included
__global__ void __launch_bounds__(256) sv_qk_rms_kernel(const KrSvAttn a) {
    __shared__ float red[4];
    const int t = blockIdx.x, part = blockIdx.y;
    const int n = (part ? a.kv_heads : a.heads) * a.dim;
    const float* z = a.qkv + (size_t)t * a.ldq + (part ? a.heads * a.dim : 0);
    const float* b = part ? a.k_bias : a.q_bias;
    float q = 0.0f;
    for (int c = threadIdx.x; c < n; c += 256) { const float v = b ? z[c] + b[c] : z[c]; q = __builtin_fmaf(v, v, q); }
    q = sv_block_sum<4>(q, red);
    if (threadIdx.x == 0) a.inv_rms_out[(size_t)t * 2 + part] = 1.0f / sqrtf(q / (float)n + a.eps);
}

// one wave per (token, head): the head vector is staged in LDS, rotated and normed there; q heads are written back in place, k heads go to the
// cache page of (slot, position), v heads are copied there
__device__ __forceinline__ void sv_wave_sync() { __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront"); __builtin_amdgcn_wave_barrier(); __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront"); }
template <typename T>
__device__ __forceinline__ void sv_qk_prep_row(const KrSvAttn& a, const int t, const int hh, const int lane, float* hv /* [dim], the wave's own */) {
    const int H = a.heads, G = a.kv_heads;
    const int p = a.pos[t], sl = a.slot[t];
    float* row = a.qkv + (size_t)t * a.ldq;
    size_t prow = 0;
    if (hh >= H) {
        const size_t page = (size_t)a.page_table[(size_t)sl * a.table_ld + p / a.page_tokens];
        prow = page * a.page_tokens + (p % a.page_tokens);
    }
    if (hh >= H + G) {                       // value head (never launched when the values are the keys): copy, or blend with the values an earlier layer formed for this token
        const int g = hh - H - G;
        const float* v = row + (size_t)H * a.dim + (size_t)G * a.dim + (size_t)g * a.vdim;
        T* dst = (T*)a.vpool + prow * a.ldv + (size_t)g * a.vdim;
        float* vf = a.v_mix ? a.v_first + ((size_t)t * G + g) * a.vdim : nullptr;
        const float lam = a.v_mix == 2 ? *a.v_lambda : 0.0f;
        const float* vb = a.v_bias ? a.v_bias + (size_t)g * a.vdim : nullptr;
        for (int d = lane; d < a.vdim; d += 64) {
            float val = vb ? v[d] + vb[d] : v[d];
            if (a.v_mix == 1) vf[d] = val;
            else if (a.v_mix == 2) val = (1.0f - lam) * val + lam * vf[d];
            sv_st(dst + d, val);
        }
        return;
    }
    float* v = row + (size_t)hh * a.dim;
    {
        const float* bias = hh < H ? a.q_bias : a.k_bias;
        if (bias) bias += (size_t)(hh < H ? hh : hh - H) * a.dim;
        for (int d = lane; d < a.dim; d += 64) hv[d] = bias ? v[d] + bias[d] : v[d];
    }
    sv_wave_sync();
    if (a.v_from_k && hh >= H) {             // the value row of this key head: the key as projected
        T* dst = (T*)a.vpool + prow * a.ldv + (size_t)(hh - H) * a.dim;
        for (int d = lane; d < a.dim; d += 64) sv_st(dst + d, hv[d]);
    }
    if (a.unit_norm == 3) {                  // one statistic for the whole row, a weight per coordinate of the row
        const float inv3 = a.inv_rms[(size_t)t * 2 + (hh < H ? 0 : 1)];
        const float* w = hh < H ? a.q_norm_w + (size_t)hh * a.dim : a.k_norm_w + (size_t)(hh - H) * a.dim;
        for (int d = lane; d < a.dim; d += 64) hv[d] = hv[d] * inv3 * w[d];
        sv_wave_sync();
    }
    if (a.unit_norm == 2) {                  // weighted, before the rotation
        const float* w = hh < H ? a.q_norm_w : a.k_norm_w;
        float s2 = 0.0f;
        for (int d = lane; d < a.dim; d += 64) s2 = __builtin_fmaf(hv[d], hv[d], s2);
        s2 = sv_wave_sum(s2);
        const float inv2 = 1.0f / sqrtf(s2 / (float)a.dim + a.eps);
        for (int d = lane; d < a.dim; d += 64) hv[d] = hv[d] * inv2 * w[d];
        sv_wave_sync();
    }
    const int half = a.rot_dims / 2;
    const float2* cs = a.cs + (size_t)t * half;
    float ss = 0.0f;
    for (int i = lane; i < half; i += 64) {  // a lane owns whole rotation pairs; the tail past rot_dims passes unchanged
        const int i0 = a.rot_interleaved ? 2 * i : i, i1 = a.rot_interleaved ? 2 * i + 1 : i + half;
        const float u = hv[i0], w = hv[i1];
        const float2 c = cs[i];
        const float r0 = u * c.x - w * c.y, r1 = w * c.x + u * c.y;
        hv[i0] = r0; hv[i1] = r1;
        ss = __builtin_fmaf(r0, r0, ss); ss = __builtin_fmaf(r1, r1, ss);
    }
    for (int d = a.rot_dims + lane; d < a.dim; d += 64) ss = __builtin_fmaf(hv[d], hv[d], ss);
    ss = sv_wave_sum(ss);
    const float inv = a.unit_norm == 1 ? 1.0f / sqrtf(ss / (float)a.dim + a.eps) : 1.0f;
    sv_wave_sync();
    if (hh < H) {
        for (int d = lane; d < a.dim; d += 64) v[d] = hv[d] * inv;
    } else {
        const int g = hh - H;
        T* dst = (T*)a.kpool + prow * a.ldk + (size_t)g * a.dim;
        for (int d = lane; d < a.dim; d += 64) sv_st(dst + d, hv[d] * inv);
    }
}
template <typename T>
__global__ void __launch_bounds__(64) sv_qk_prep_kernel(const KrSvAttn a) {
    extern __shared__ float hv[];            // [dim]
    sv_qk_prep_row<T>(a, blockIdx.x, blockIdx.y, threadIdx.x, hv);
}

// Windowed attention with a sink over the paged cache.  One workgroup (four waves) per (token, key / value head, batch of RM query heads of that
// head's group): a cache row is fetched once for all query heads that share it.  The visible keys [max(0, p - window + 1), p] are walked in blocks of
// 64, block b by wave b % 4; lane j scores key j for every head (f32 dot of the pre-scaled query, held in LDS, with the 16-byte pieces of its key row),
// the wave updates each head's running maximum / denominator (online softmax, f32) and the lanes then own value columns for p.v.  The four waves'
// partial states are merged through LDS in wave order; the sink joins the denominator there, once.
typedef uint32_t sv_u4 __attribute__((ext_vector_type(4)));
#ifdef KR_SV_STAMPS      // probe build: shader-clock stamps of the first wave of the first workgroup (kr_sv_read_stamps)
__device__ long long sv_stamps[16];
#define SV_STAMP(i) do { if (blockIdx.x == 0 && blockIdx.y == 0 && blockIdx.z == 0 && threadIdx.x == 0) sv_stamps[i] = __builtin_readcyclecounter(); } while (0)
#else
#define SV_STAMP(i) do { } while (0)
#endif
template <typename T, int RM, int VC>
__global__ void __launch_bounds__(256) sv_attn_group_kernel(const KrSvAttn a) {
    extern __shared__ __attribute__((aligned(16))) float lds[];
    constexpr int VEC = 16 / sizeof(T);
    const int G = a.kv_heads, R = a.heads / G, dim = a.dim, vdim = a.vdim;
    const int sp = blockIdx.z % a.nsplit;
    const int t = blockIdx.x, g = blockIdx.y, r0 = (blockIdx.z / a.nsplit) * RM, nr = min(RM, R - r0), h0 = g * R + r0;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    float* qs = lds;                                       // [RM][dim]
    float* pw = qs + RM * dim + wave * 64 * RM;            // this wave's weights [RM][64]
    float* ml = qs + RM * dim + 4 * 64 * RM;               // [4][RM][2]
    float* accs = ml + 4 * RM * 2;                         // [RM][vdim]
    const int p = a.pos[t], sl = a.slot[t];
    const int* table = a.page_table + (size_t)sl * a.table_ld;
    const float* q = a.qkv + (size_t)t * a.ldq + (size_t)h0 * dim;
    // heads past the group's last one are computed on zero queries and dropped: the loops below carry no per-head branches, so the loads of a block of
    // keys are all in flight before the first product needs them
    SV_STAMP(0);
    for (int i = tid; i < RM * dim; i += 256) qs[i] = i < nr * dim ? q[i] * a.scale : 0.0f;
    __syncthreads();
    SV_STAMP(1);
    int lo = a.window > 0 ? max(0, p - a.window + 1) : (a.chunk > 0 ? p - p % a.chunk : 0);
    // kept first keys: their own leading blocks when the window has left them behind, else one contiguous range from 0
    const int nck = a.keep > 0 && lo > a.keep ? (a.keep + 63) / 64 : 0;
    if (a.keep > 0 && nck == 0) lo = 0;
    float slope[RM];
#pragma unroll
    for (int r = 0; r < RM; r++) slope[r] = (a.slopes && r < nr) ? a.slopes[h0 + r] : 0.0f;
    float m[RM], l[RM], acc[RM][VC];
#pragma unroll
    for (int r = 0; r < RM; r++) {
        m[r] = -INFINITY; l[r] = 0.0f;
#pragma unroll
        for (int c = 0; c < VC; c++) acc[r][c] = 0.0f;
    }
    const T* kp = (const T*)a.kpool; const T* vp = (const T*)a.vpool;
    const bool vec = ((size_t)dim * sizeof(T)) % 16 == 0 && ((size_t)a.ldk * sizeof(T)) % 16 == 0;
    const int npiece = dim / VEC;
    auto widen = [](const sv_u4& kv, float* kf) {
        if constexpr (sizeof(T) == 2) {
#pragma unroll
            for (int i = 0; i < 4; i++) { kf[2 * i] = __uint_as_float(kv[i] << 16); kf[2 * i + 1] = __uint_as_float(kv[i] & 0xFFFF0000u); }
        } else {
#pragma unroll
            for (int i = 0; i < 4; i++) kf[i] = __uint_as_float(kv[i]);
        }
    };
    // blocks of 64 keys: this workgroup's share [c0, c1) of the token's blocks (all of them when the launch is not split), block c by wave (c - c0) % 4
    const int nch = (p - lo) / 64 + 1 + nck, cps = (nch + a.nsplit - 1) / a.nsplit;
    const int c0 = sp * cps, c1 = min(nch, c0 + cps);
    for (int cb = c0 + wave; cb < c1; cb += 4) {
        const int j0 = cb < nck ? 64 * cb : lo + 64 * (cb - nck), jl = cb < nck ? a.keep - 1 : p;
        const int j = j0 + lane;
        const bool live = j <= jl;
        const int jc = min(j, jl);                           // lanes past the last key score it again; their weight is set to 0
        const int prow = table[jc / a.page_tokens] * a.page_tokens + (jc % a.page_tokens);
        const T* k = kp + (size_t)prow * a.ldk + (size_t)g * dim;
        constexpr int U = 16 / VC;                           // keys whose value rows are requested together
        const int nk = min(64, jl - j0 + 1);
        float va[U][VC], vb[U][VC];
        auto fetch_v = [&](int jb, float (&vv)[U][VC]) {
#pragma unroll
            for (int u = 0; u < U; u++) {
                const int pr = __builtin_amdgcn_readlane(prow, min(jb + u, 63));
                const T* vr = vp + (size_t)pr * a.ldv + (size_t)g * vdim;
#pragma unroll
                for (int c = 0; c < VC; c++) { const int d = lane + 64 * c; vv[u][c] = d < vdim ? sv_ld(vr + d) : 0.0f; }
            }
        };
        SV_STAMP(2);
        fetch_v(0, va);                                      // in flight behind the key rows, consumed after the softmax
        float s[RM];
#pragma unroll
        for (int r = 0; r < RM; r++) s[r] = 0.0f;
        if (vec) {
            int pc = 0;
            auto block = [&](auto PBc) {                     // PB 16-byte pieces of the key row in flight, then their products with every head's query
                constexpr int PB = decltype(PBc)::value;
                sv_u4 kv[PB];
#pragma unroll
                for (int u = 0; u < PB; u++) kv[u] = *reinterpret_cast<const sv_u4*>(k + (pc + u) * VEC);
#pragma unroll
                for (int u = 0; u < PB; u++) {
                    float kf[VEC];
                    widen(kv[u], kf);
#pragma unroll
                    for (int r = 0; r < RM; r++) {
                        const float4* qp = reinterpret_cast<const float4*>(qs + r * dim + (pc + u) * VEC);
#pragma unroll
                        for (int v4 = 0; v4 < VEC / 4; v4++) {
                            const float4 qa = qp[v4];
                            s[r] = __builtin_fmaf(qa.x, kf[4 * v4], s[r]); s[r] = __builtin_fmaf(qa.y, kf[4 * v4 + 1], s[r]);
                            s[r] = __builtin_fmaf(qa.z, kf[4 * v4 + 2], s[r]); s[r] = __builtin_fmaf(qa.w, kf[4 * v4 + 3], s[r]);
                        }
                    }
                }
                pc += PB;
            };
            while (pc + 16 <= npiece) block(std::integral_constant<int, 16>{});
            if (pc + 8 <= npiece) block(std::integral_constant<int, 8>{});
            if (pc + 4 <= npiece) block(std::integral_constant<int, 4>{});
            for (; pc < npiece; pc++) {
                const sv_u4 kv = *reinterpret_cast<const sv_u4*>(k + pc * VEC);
                float kf[VEC];
                widen(kv, kf);
#pragma unroll
                for (int r = 0; r < RM; r++)
#pragma unroll
                    for (int i = 0; i < VEC; i++) s[r] = __builtin_fmaf(qs[r * dim + pc * VEC + i], kf[i], s[r]);
            }
        } else {
            for (int d = 0; d < dim; d++) {
                const float kd = sv_ld(k + d);
#pragma unroll
                for (int r = 0; r < RM; r++) s[r] = __builtin_fmaf(qs[r * dim + d], kd, s[r]);
            }
        }
        SV_STAMP(3);
#pragma unroll
        for (int r = 0; r < RM; r++) {
            const float sc = a.softcap > 0.0f ? a.softcap * tanhf(s[r] / a.softcap) : s[r];
            const float sr = live ? sc - slope[r] * (float)(p - j) : -INFINITY;
            const float mn = fmaxf(m[r], sv_wave_max(sr));
            const float alpha = expf(m[r] - mn);               // first block of this wave: exp(-inf) = 0
            const float pj = live ? expf(sr - mn) : 0.0f;
            l[r] = l[r] * alpha + sv_wave_sum(pj);
            m[r] = mn;
#pragma unroll
            for (int c = 0; c < VC; c++) acc[r][c] *= alpha;
            pw[r * 64 + lane] = pj;
        }
        // the wave's own LDS writes are read back by its own lanes below: a wave executes in lock step, only the LDS counter has to drain
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        SV_STAMP(4);
        // groups of U keys: a group's products run while the next group's value rows are in flight (the first group's were requested before the scores);
        // keys past nk inside the last group carry weight 0 and read the last key's row
        auto products = [&](int jb, float (&vv)[U][VC]) {
#pragma unroll
            for (int r = 0; r < RM; r++) {
                if constexpr (U % 4 == 0) {      // four keys' weights per LDS read (jb is a multiple of U: the read is 16-byte aligned and stays inside the block)
#pragma unroll
                    for (int u4 = 0; u4 < U / 4; u4++) {
                        const float4 w4 = *reinterpret_cast<const float4*>(&pw[r * 64 + jb + 4 * u4]);
#pragma unroll
                        for (int c = 0; c < VC; c++) {
                            acc[r][c] = __builtin_fmaf(w4.x, vv[4 * u4][c], acc[r][c]); acc[r][c] = __builtin_fmaf(w4.y, vv[4 * u4 + 1][c], acc[r][c]);
                            acc[r][c] = __builtin_fmaf(w4.z, vv[4 * u4 + 2][c], acc[r][c]); acc[r][c] = __builtin_fmaf(w4.w, vv[4 * u4 + 3][c], acc[r][c]);
                        }
                    }
                } else {
#pragma unroll
                    for (int u = 0; u < U; u++) {
                        const float w = pw[r * 64 + min(jb + u, 63)];
#pragma unroll
                        for (int c = 0; c < VC; c++) acc[r][c] = __builtin_fmaf(w, vv[u][c], acc[r][c]);
                    }
                }
            }
        };
        for (int jb = 0; jb < nk; jb += 2 * U) {
            if (jb + U < nk) fetch_v(jb + U, vb);
            products(jb, va);
            if (jb + 2 * U < nk) fetch_v(jb + 2 * U, va);
            if (jb + U < nk) products(jb + U, vb);
        }
        SV_STAMP(5);
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    }
    if (lane == 0) {
#pragma unroll
        for (int r = 0; r < RM; r++) if (r < nr) { ml[(wave * RM + r) * 2] = m[r]; ml[(wave * RM + r) * 2 + 1] = l[r]; }
    }
    __syncthreads();
    SV_STAMP(6);
    const bool last = a.nsplit == 1;                         // an unsplit launch finishes here: sink, normalisation, output; a split one leaves partial states
    float f[RM];
#pragma unroll
    for (int r = 0; r < RM; r++) {
        f[r] = 0.0f;
        if (r < nr) {
            float M = -INFINITY;
            for (int w = 0; w < 4; w++) M = fmaxf(M, ml[(w * RM + r) * 2]);
            if (last && a.sink) M = fmaxf(M, a.sink[h0 + r]);
            f[r] = m[r] == -INFINITY ? 0.0f : expf(m[r] - M);
        }
    }
    for (int w = 0; w < 4; w++) {
        if (wave == w) {
#pragma unroll
            for (int r = 0; r < RM; r++) {
                if (r < nr) {
#pragma unroll
                    for (int c = 0; c < VC; c++) {
                        const int d = lane + 64 * c;
                        if (d < vdim) accs[r * vdim + d] = (w == 0 ? 0.0f : accs[r * vdim + d]) + acc[r][c] * f[r];
                    }
                }
            }
        }
        __syncthreads();
    }
    T* o = (T*)a.out + (size_t)t * (a.out_ld ? a.out_ld : a.heads * vdim) + (size_t)h0 * vdim;
    const float osc = a.out_scale != 0.0f ? a.out_scale : 1.0f;
    for (int i = tid; i < nr * vdim; i += 256) {
        const int r = i / vdim;
        float M = -INFINITY;
        for (int w = 0; w < 4; w++) M = fmaxf(M, ml[(w * RM + r) * 2]);
        if (last && a.sink) M = fmaxf(M, a.sink[h0 + r]);
        float L = (last && a.sink) ? expf(a.sink[h0 + r] - M) : 0.0f;
        for (int w = 0; w < 4; w++) { const float mw = ml[(w * RM + r) * 2]; if (mw != -INFINITY) L += ml[(w * RM + r) * 2 + 1] * expf(mw - M); }
        if (last) {
            const float gt = a.out_gate ? 1.0f / (1.0f + expf(-a.out_gate[(size_t)t * a.ld_gate + (a.gate_elem ? (size_t)h0 * vdim + i : (size_t)(h0 + r))])) : 1.0f;
            sv_st(o + i, accs[i] / L * gt * osc);
        }
        else {
            const size_t slot = ((size_t)t * a.heads + h0 + r) * a.nsplit + sp;
            a.part_acc[slot * vdim + (i - r * vdim)] = accs[i];
            if (i == r * vdim) { a.part_ml[slot * 2] = M; a.part_ml[slot * 2 + 1] = L; }
        }
    }
    SV_STAMP(7);
}

// Prompt-sized steps: the same attention on the f32 matrix instruction (v_mfma_f32_16x16x4_f32: every product and sum stays f32).  A workgroup owns 16
// query ROWS that share one key / value head -- the heads of its group for one token, or for 16 / R consecutive tokens of one request when the group has
// fewer than 16 heads (a row carries its own position, so the causal and window masks are per row) -- and its four waves split the blocks of 64 keys.
// Both products are formed TRANSPOSED so that nothing is shuffled between them:
//   S^T[key][row] = K Q^T   (A = key rows, B = the rows' queries, held in registers for the whole launch)
//   O^T[d][row]  += V^T P^T (A = value columns, B = the weights exactly where the first product left them: lane = row, register = key)
// so a lane's accumulators all belong to ONE row and the online-softmax rescale is a per-lane scalar.  The reduction index of an MFMA is spread over the
// four 16-lane groups; group q takes the CONTIGUOUS quarter q of a key row (dim / 4 elements, 16-byte loads) and the keys 4 q .. 4 q + 3 of a 16-key block.
typedef float sv_f4 __attribute__((ext_vector_type(4)));
template <typename T, int DQ, int DB, int NKB = 4>      // DQ = dim / 4 query elements per lane, DB = vdim / 16 value columns per lane, NKB = blocks of 16 keys a wave takes at a time
__global__ void __launch_bounds__(256) sv_attn_mfma_kernel(const KrSvAttn a) {
    extern __shared__ __attribute__((aligned(16))) float lds[];
    constexpr int VEC = 16 / sizeof(T);
    const int G = a.kv_heads, R = a.heads / G, dim = DQ * 4, vdim = DB * 16;
    const int Rb = R < 16 ? R : 16, TQ = a.tq;             // tokens per workgroup: 16 / Rb for prompt portions, 1 for decode-shaped steps (rows past TQ * Rb idle)
    const int sp = blockIdx.z % a.nsplit, hb = blockIdx.z / a.nsplit;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, row = lane & 15, qd = lane >> 4;
    const int g = blockIdx.y, h_row = g * R + hb * 16 + (row % Rb), t0 = blockIdx.x * TQ, tq_row = row / Rb;
    float* ml = lds;                    // [4 waves][16 rows][2]
    float* mf = lds + 4 * 16 * 2;       // [16 rows][2]: the merged maximum and 1 / denominator (or the denominator itself in a split launch)
    // [16 rows][AS]: a row is vdim + 65 floats long and the column block of lane group qd starts 16 floats late, so that the 64 lanes of a wave, which hold the
    // same column of 16 rows x 4 groups, fall into distinct LDS banks (rows of exactly vdim floats put all of them into ONE bank)
    float* accs = mf + 16 * 2;
    constexpr int AS = DB * 16 + 65;
    auto acc_at = [](int r, int c) { return r * AS + c + (c / (4 * DB)) * 16; };
    const T* kp = (const T*)a.kpool; const T* vp = (const T*)a.vpool;
    for (int base = 0; base < TQ && t0 + base < a.T;) {
        // the run of tokens [base, end) of this group that continue one request (same slot, consecutive positions)
        const int sl = a.slot[t0 + base], p0 = a.pos[t0 + base];
        int end = base + 1;
        while (end < TQ && t0 + end < a.T && a.slot[t0 + end] == sl && a.pos[t0 + end] == p0 + (end - base)) end++;
        const bool rv = tq_row >= base && tq_row < end;
        const int p_row = rv ? p0 + (tq_row - base) : -1;
        const int lo_row = a.window > 0 ? max(0, p_row - a.window + 1) : (a.chunk > 0 && rv ? p_row - p_row % a.chunk : 0);
        const int hi = p0 + (end - base - 1);
        int lo = a.window > 0 ? max(0, p0 - a.window + 1) : (a.chunk > 0 ? p0 - p0 % a.chunk : 0);
        const int keep_row = rv ? a.keep : 0;
        const float slope_row = (a.slopes && rv) ? a.slopes[h_row] : 0.0f;
        const int* table = a.page_table + (size_t)sl * a.table_ld;
        float q[DQ];
        {
            const float* qp = a.qkv + (size_t)(t0 + (rv ? tq_row : base)) * a.ldq + (size_t)h_row * dim + qd * DQ;
#pragma unroll
            for (int i = 0; i < DQ; i++) q[i] = rv ? qp[i] * a.scale : 0.0f;
        }
        float m = -INFINITY, l = 0.0f;
        sv_f4 acc[DB];
#pragma unroll
        for (int d = 0; d < DB; d++) acc[d] = sv_f4{0.0f, 0.0f, 0.0f, 0.0f};
        constexpr int KEYS = 16 * NKB;
        // kept first keys: their own leading blocks when every row's window has left them behind, else one contiguous range from 0
        const int nck = a.keep > 0 && lo > a.keep ? (a.keep + KEYS - 1) / KEYS : 0;
        if (a.keep > 0 && nck == 0) lo = 0;
        const int nch = (hi - lo) / KEYS + 1 + nck, cps = (nch + a.nsplit - 1) / a.nsplit, c0 = sp * cps, c1 = min(nch, c0 + cps);
        for (int cb = c0 + wave; cb < c1; cb += 4) {
            const int j0 = cb < nck ? KEYS * cb : lo + KEYS * (cb - nck), jl = cb < nck ? a.keep - 1 : hi;
            // ---- S^T: NKB blocks of 16 keys
            sv_f4 st[NKB];
            int prow[NKB];
#pragma unroll
            for (int kb = 0; kb < NKB; kb++) {
                const int key = min(j0 + kb * 16 + row, jl);         // keys past the last one are fetched again and masked
                prow[kb] = table[key / a.page_tokens] * a.page_tokens + (key % a.page_tokens);
            }
#pragma unroll
            for (int kb = 0; kb < NKB; kb++) {
                const T* k = kp + (size_t)prow[kb] * a.ldk + (size_t)g * dim + qd * DQ;
                // a key row's quarter in batches of at most PB 16-byte pieces: long rows (a latent cache row) must not hold all of it in registers at once
                constexpr int NP = DQ / VEC, PB = NP <= 8 ? NP : 6;
                sv_f4 c = sv_f4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
                for (int u0 = 0; u0 < NP; u0 += PB) {
                    sv_u4 kv[PB];
#pragma unroll
                    for (int u = 0; u < PB; u++) if (u0 + u < NP) kv[u] = *reinterpret_cast<const sv_u4*>(k + (u0 + u) * VEC);
#pragma unroll
                    for (int u = 0; u < PB; u++) {
                        if (u0 + u >= NP) continue;
                        float kf[VEC];
                        if constexpr (sizeof(T) == 2) {
#pragma unroll
                            for (int i = 0; i < 4; i++) { kf[2 * i] = __uint_as_float(kv[u][i] << 16); kf[2 * i + 1] = __uint_as_float(kv[u][i] & 0xFFFF0000u); }
                        } else {
#pragma unroll
                            for (int i = 0; i < 4; i++) kf[i] = __uint_as_float(kv[u][i]);
                        }
#pragma unroll
                        for (int i = 0; i < VEC; i++) c = __builtin_amdgcn_mfma_f32_16x16x4f32(kf[i], q[(u0 + u) * VEC + i], c, 0, 0, 0);
                    }
                }
                st[kb] = c;
            }
            // ---- masks and the online softmax of this lane's row (its 16 keys here, the other 48 in the three lanes 16 apart)
            float cm = -INFINITY;
#pragma unroll
            for (int kb = 0; kb < NKB; kb++)
#pragma unroll
                for (int i = 0; i < 4; i++) {
                    const int key = j0 + kb * 16 + 4 * qd + i;
                    const bool ok = rv && key <= min(p_row, jl) && (key >= lo_row || key < keep_row);
                    const float sc = a.softcap > 0.0f ? a.softcap * tanhf(st[kb][i] / a.softcap) : st[kb][i];
                    st[kb][i] = ok ? sc - slope_row * (float)(p_row - key) : -INFINITY;
                    cm = fmaxf(cm, st[kb][i]);
                }
            cm = fmaxf(cm, __shfl_xor(cm, 16)); cm = fmaxf(cm, __shfl_xor(cm, 32));
            const float mn = fmaxf(m, cm);
            const float alpha = mn == -INFINITY ? 1.0f : expf(m - mn);       // a row that has seen no key yet keeps its zero state
            float ps = 0.0f;
#pragma unroll
            for (int kb = 0; kb < NKB; kb++)
#pragma unroll
                for (int i = 0; i < 4; i++) { const float pj = st[kb][i] == -INFINITY ? 0.0f : expf(st[kb][i] - mn); st[kb][i] = pj; ps += pj; }
            ps += __shfl_xor(ps, 16); ps += __shfl_xor(ps, 32);
            l = l * alpha + ps; m = mn;
#pragma unroll
            for (int d = 0; d < DB; d++) acc[d] *= alpha;
            // ---- O^T += V^T P^T: key (kb, 4 qd + i) -> this lane reads its DB value columns of that key's row
            // wide values (DB > 16) go through in column batches of DC, so that one batch of four keys' values is in registers at a time
            constexpr int DC = DB <= 16 ? DB : 8;
#pragma unroll
            for (int kb = 0; kb < NKB; kb++) {
                int prk[4];
#pragma unroll
                for (int i = 0; i < 4; i++) prk[i] = __shfl(prow[kb], 4 * qd + i);
#pragma unroll
                for (int d0 = 0; d0 < DB; d0 += DC) {
                    float vf[4][DC];
#pragma unroll
                    for (int i = 0; i < 4; i++) {
                        const T* vr = vp + (size_t)prk[i] * a.ldv + (size_t)g * vdim + row * DB + d0;
                        if constexpr ((DC * sizeof(T)) % 16 == 0 && (DB * sizeof(T)) % 16 == 0) {
#pragma unroll
                            for (int u = 0; u < DC / VEC; u++) {
                                const sv_u4 vv = *reinterpret_cast<const sv_u4*>(vr + u * VEC);
                                if constexpr (sizeof(T) == 2) {
#pragma unroll
                                    for (int e = 0; e < 4; e++) { vf[i][u * VEC + 2 * e] = __uint_as_float(vv[e] << 16); vf[i][u * VEC + 2 * e + 1] = __uint_as_float(vv[e] & 0xFFFF0000u); }
                                } else {
#pragma unroll
                                    for (int e = 0; e < 4; e++) vf[i][u * VEC + e] = __uint_as_float(vv[e]);
                                }
                            }
                        } else {
#pragma unroll
                            for (int e = 0; e < DC; e++) vf[i][e] = sv_ld(vr + e);
                        }
                    }
#pragma unroll
                    for (int i = 0; i < 4; i++)
#pragma unroll
                        for (int d = 0; d < DC; d++) acc[d0 + d] = __builtin_amdgcn_mfma_f32_16x16x4f32(vf[i][d], st[kb][i], acc[d0 + d], 0, 0, 0);
                }
            }
        }
        // ---- the four waves' states -> one, in wave order; an unsplit launch adds the sink and writes the output, a split one leaves (maximum, denominator, sums)
        const bool last = a.nsplit == 1;
        __syncthreads();
        if (qd == 0) { ml[(wave * 16 + row) * 2] = m; ml[(wave * 16 + row) * 2 + 1] = l; }
        __syncthreads();
        if (tid < 16) {
            const int h = g * R + hb * 16 + (tid % Rb);
            float Mr = -INFINITY;
            for (int w = 0; w < 4; w++) Mr = fmaxf(Mr, ml[(w * 16 + tid) * 2]);
            if (last && a.sink) Mr = fmaxf(Mr, a.sink[h]);
            float L = (last && a.sink) ? expf(a.sink[h] - Mr) : 0.0f;
            for (int w = 0; w < 4; w++) { const float mw = ml[(w * 16 + tid) * 2]; if (mw != -INFINITY) L += ml[(w * 16 + tid) * 2 + 1] * expf(mw - Mr); }
            mf[tid * 2] = Mr; mf[tid * 2 + 1] = last ? 1.0f / L : L;
        }
        __syncthreads();
        const float f = m == -INFINITY ? 0.0f : expf(m - mf[row * 2]);
        for (int w = 0; w < 4; w++) {
            if (wave == w) {
#pragma unroll
                for (int d = 0; d < DB; d++)
#pragma unroll
                    for (int i = 0; i < 4; i++) {
                        const int col = (4 * qd + i) * DB + d;
                        accs[acc_at(row, col)] = (w == 0 ? 0.0f : accs[acc_at(row, col)]) + acc[d][i] * f;
                    }
            }
            __syncthreads();
        }
        for (int i = tid; i < 16 * vdim; i += 256) {
            const int r = i / vdim, tq = r / Rb;
            if (tq < base || tq >= end) continue;
            const int h = g * R + hb * 16 + (r % Rb);
            const float av = accs[acc_at(r, i - r * vdim)];
            if (last) {
                const float gt = a.out_gate ? 1.0f / (1.0f + expf(-a.out_gate[(size_t)(t0 + tq) * a.ld_gate + (a.gate_elem ? (size_t)h * vdim + (i - r * vdim) : (size_t)h)])) : 1.0f;
                sv_st((T*)a.out + (size_t)(t0 + tq) * (a.out_ld ? a.out_ld : a.heads * vdim) + (size_t)h * vdim + (i - r * vdim), av * mf[r * 2 + 1] * gt * (a.out_scale != 0.0f ? a.out_scale : 1.0f));
            }
            else {
                const size_t slot = ((size_t)(t0 + tq) * a.heads + h) * a.nsplit + sp;
                a.part_acc[slot * vdim + (i - r * vdim)] = av;
                if (i == r * vdim) { a.part_ml[slot * 2] = mf[r * 2]; a.part_ml[slot * 2 + 1] = mf[r * 2 + 1]; }
            }
        }
        __syncthreads();
        base = end;
    }
}

// the partial states of a split launch -> output: one workgroup per (token, head).  The splits' weights exp(m_s - M) are formed once (LDS); a thread then owns
// value columns and its loads over the splits do not depend on one another
template <typename T>
__global__ void __launch_bounds__(256) sv_attn_merge_kernel(const KrSvAttn a) {
    extern __shared__ float wsp[];           // [nsplit] weight of every split, then 1 / denominator
    const int t = a.toks ? a.toks[blockIdx.x] : (int)blockIdx.x, h = blockIdx.y, tid = threadIdx.x;
    const size_t base = ((size_t)(a.form == KR_SV_ATTN_STEP ? blockIdx.x : t) * a.heads + h) * a.nsplit;
    const float sink = a.sink ? (a.form ? a.sink[h] * 1.44269504f : a.sink[h]) : -INFINITY;      // the split forms keep their maxima in powers of two
    auto ex = [&](float x) { return a.form ? exp2f(x) : expf(x); };
    float M = sink;
    for (int s = 0; s < a.nsplit; s++) M = fmaxf(M, a.part_ml[(base + s) * 2]);
    for (int s = tid; s < a.nsplit; s += 256) { const float ms = a.part_ml[(base + s) * 2]; wsp[s] = ms == -INFINITY ? 0.0f : ex(ms - M); }
    __syncthreads();
    if (tid == 0) {
        float L = a.sink ? ex(sink - M) : 0.0f;
        for (int s = 0; s < a.nsplit; s++) if (wsp[s] != 0.0f) L = __builtin_fmaf(a.part_ml[(base + s) * 2 + 1], wsp[s], L);
        wsp[a.nsplit] = 1.0f / L;
    }
    __syncthreads();
    const float inv = wsp[a.nsplit] * ((a.out_gate && !a.gate_elem) ? 1.0f / (1.0f + expf(-a.out_gate[(size_t)t * a.ld_gate + h])) : 1.0f) * (a.out_scale != 0.0f ? a.out_scale : 1.0f);
    T* o = (T*)a.out + (size_t)t * (a.out_ld ? a.out_ld : a.heads * a.vdim) + (size_t)h * a.vdim;
    for (int d = tid; d < a.vdim; d += 256) {
        float v = 0.0f;
#pragma unroll 8
        for (int s = 0; s < a.nsplit; s++) { const float w = wsp[s], p = a.part_acc[(base + s) * a.vdim + d]; v = __builtin_fmaf(w != 0.0f ? p : 0.0f, w, v); }      // a split without keys counts as zeros
        if (a.out_gate && a.gate_elem) v *= 1.0f / (1.0f + expf(-a.out_gate[(size_t)t * a.ld_gate + (size_t)h * a.vdim + d]));
        sv_st(o + d, v * inv);
    }
}

// selection: one wave per token; the scores of the E experts live in LDS
// z holds the logits as `parts` column blocks of E that are added (a gate stored as two bf16 terms gives two)
__global__ void __launch_bounds__(64) sv_router_select_kernel(const float* __restrict__ z, int ld, int parts, const float* __restrict__ bias, int bias_mode, int score_kind,
                                                              int group_kind, int E, int top, int groups, int keep, int renorm, int* __restrict__ ids, float* __restrict__ wts) {
    extern __shared__ float lds[];           // s[E] scores | c[E] choice scores | gscore[groups] | allowed flags as floats [groups]
    float* s = lds; float* cs = lds + E; float* gs = cs + E; float* gok = gs + groups;
    const int t = blockIdx.x, lane = threadIdx.x;
    for (int e = lane; e < E; e += 64) {
        float v = z[(size_t)t * ld + e];
        for (int q = 1; q < parts; q++) v += z[(size_t)t * ld + (size_t)q * E + e];
        s[e] = (bias && bias_mode == 1) ? v + bias[e] : v;
    }
    __syncthreads();
    if (score_kind == 1) {
        for (int e = lane; e < E; e += 64) s[e] = 1.0f / (1.0f + expf(-s[e]));
    } else {
        float mx = -INFINITY;
        for (int e = lane; e < E; e += 64) mx = fmaxf(mx, s[e]);
        mx = sv_wave_max(mx);
        float sum = 0.0f;
        for (int e = lane; e < E; e += 64) { const float v = expf(s[e] - mx); s[e] = v; sum += v; }
        __syncthreads();
        sum = sv_wave_sum(sum);
        const float inv = 1.0f / sum;
        for (int e = lane; e < E; e += 64) s[e] *= inv;
    }
    for (int e = lane; e < E; e += 64) cs[e] = (bias && bias_mode == 2) ? s[e] + bias[e] : s[e];
    __syncthreads();
    const int per = E / groups;
    for (int gi = lane; gi < groups; gi += 64) {
        float v = -INFINITY, v2 = -INFINITY;       // the two largest of the group
        for (int e = gi * per; e < (gi + 1) * per; e++) { const float c = cs[e]; if (c > v) { v2 = v; v = c; } else if (c > v2) v2 = c; }
        gs[gi] = (group_kind == 1 && per > 1) ? v + v2 : v; gok[gi] = groups == keep ? 1.0f : 0.0f;
    }
    __syncthreads();
    if (keep < groups) {
        for (int r = 0; r < keep; r++) {         // r-th best group: largest score, lowest index among equals
            float bv = -INFINITY; int bi = 0x7fffffff;
            for (int gi = lane; gi < groups; gi += 64) if (gok[gi] == 0.0f && (gs[gi] > bv || (gs[gi] == bv && gi < bi))) { bv = gs[gi]; bi = gi; }
#pragma unroll
            for (int o = 32; o > 0; o >>= 1) {
                const float ov = __shfl_xor(bv, o); const int oi = __shfl_xor(bi, o);
                if (ov > bv || (ov == bv && oi < bi)) { bv = ov; bi = oi; }
            }
            __syncthreads();
            if (lane == 0 && bi != 0x7fffffff) gok[bi] = 1.0f;
            __syncthreads();
        }
    }
    float wsum = 0.0f;
    for (int r = 0; r < top; r++) {
        float bv = -INFINITY; int bi = 0x7fffffff;
        for (int e = lane; e < E; e += 64) {
            const float v = cs[e];
            if (v != -INFINITY && gok[e / per] != 0.0f && (v > bv || (v == bv && e < bi))) { bv = v; bi = e; }      // a taken expert is marked by minus infinity
        }
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) {
            const float ov = __shfl_xor(bv, o); const int oi = __shfl_xor(bi, o);
            if (ov > bv || (ov == bv && oi < bi)) { bv = ov; bi = oi; }
        }
        __syncthreads();
        float wv;
        if (bi == 0x7fffffff) { bi = 0; wv = 0.0f; }      // fewer allowed experts than `top` (refused on the host): a zero-weight slot
        else { wv = s[bi]; if (lane == 0) cs[bi] = -INFINITY; }
        if (lane == 0) { ids[(size_t)t * top + r] = bi; wts[(size_t)t * top + r] = wv; }
        wsum += wv;
        __syncthreads();
    }
    if (renorm) {
        const float rinv = 1.0f / (wsum + 1e-20f);
        for (int r = lane; r < top; r += 64) wts[(size_t)t * top + r] *= rinv;
    }
}

// Up to 128 experts: the scores of a token live in a wave's registers (NV per lane) and an expert's place among them is COUNTED -- every value is broadcast once and compared with
// all -- instead of found by `top` rounds of a wave-wide maximum, each a chain of twelve LDS shuffles and two barriers.  Same order (largest first, lowest index among equals,
// NaN and minus infinity never chosen), same sums.  SORT: a decode step's tokens are one workgroup's waves (T <= 16), which then sorts their rows by expert in the same launch.
// 64 experts, top 6: one token 12.4 + 4.7 us as two launches -> 4.0, twelve 12.8 + 4.6 -> 7.0, 4096 (choice alone) 25 -> 12.
template <int NV, bool SORT>
__device__ __forceinline__ void sv_router_rank(const KrSvRoute& ro, const int bx) {
    const float* __restrict__ z = ro.z; const float* __restrict__ bias = ro.bias;
    const int ld = ro.ld, parts = ro.parts, bias_mode = ro.bias_mode, score_kind = ro.score_kind, group_kind = ro.group_kind, T = ro.T, E = ro.E, top = ro.top, groups = ro.groups, keep = ro.keep,
              renorm = ro.renorm;
    int* __restrict__ ids = ro.ids; float* __restrict__ wts = ro.wts; int* __restrict__ seg = ro.seg; int* __restrict__ src_row = ro.src_row; int* __restrict__ row_group = ro.row_group;
    int* __restrict__ pair_pos = ro.pair_pos; float* __restrict__ row_w = ro.row_w;
    constexpr int NWAVES = SORT ? 16 : 4;
    __shared__ float gsc[NWAVES][64];                       // choice scores by expert while groups are scored (one wave's 64 at a time), then the groups' scores
    __shared__ float cho[NWAVES][64 * NV];
    __shared__ int s_ids[SORT ? 16 * 64 : 1]; __shared__ float s_w[SORT ? 16 * 64 : 1];
    __shared__ int cnt[SORT ? 128 : 1];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, t = bx * NWAVES + wave;
    if (SORT) { if (threadIdx.x < 128) cnt[threadIdx.x] = 0; }
    if (t < T) {
        float s[NV], c[NV];
#pragma unroll
        for (int i = 0; i < NV; i++) {
            const int e = lane + 64 * i;
            float v = 0.0f;
            if (e < E) {
                v = z[(size_t)t * ld + e];
                for (int q = 1; q < parts; q++) v += z[(size_t)t * ld + (size_t)q * E + e];
                if (bias && bias_mode == 1) v += bias[e];
            }
            s[i] = v;
        }
        if (score_kind == 1) {
#pragma unroll
            for (int i = 0; i < NV; i++) s[i] = 1.0f / (1.0f + expf(-s[i]));
        } else {
            float mx = -INFINITY, sum = 0.0f;
#pragma unroll
            for (int i = 0; i < NV; i++) if (lane + 64 * i < E) mx = fmaxf(mx, s[i]);
            mx = sv_wave_max(mx);
#pragma unroll
            for (int i = 0; i < NV; i++) if (lane + 64 * i < E) { s[i] = expf(s[i] - mx); sum += s[i]; }
            const float inv = 1.0f / sv_wave_sum(sum);
#pragma unroll
            for (int i = 0; i < NV; i++) s[i] *= inv;
        }
        bool ok[NV];
#pragma unroll
        for (int i = 0; i < NV; i++) {
            const int e = lane + 64 * i;
            c[i] = e < E ? ((bias && bias_mode == 2) ? s[i] + bias[e] : s[i]) : -INFINITY;
            ok[i] = e < E && c[i] == c[i] && c[i] != -INFINITY;
        }
        if (keep < groups) {                                 // only the experts of the `keep` best groups stay
            const int per = E / groups;
#pragma unroll
            for (int i = 0; i < NV; i++) cho[wave][lane + 64 * i] = c[i];
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront"); __builtin_amdgcn_wave_barrier(); __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
            float g = -INFINITY;
            if (lane < groups) {
                float v = -INFINITY, v2 = -INFINITY;         // the two largest of the group
                for (int e = lane * per; e < (lane + 1) * per; e++) { const float x = cho[wave][e]; if (x > v) { v2 = v; v = x; } else if (x > v2) v2 = x; }
                g = (group_kind == 1 && per > 1) ? v + v2 : v;
            }
            int rank = 0;
            for (int j = 0; j < groups; j++) { const float o = __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(g), j)); rank += (o > g || (o == g && j < lane)) ? 1 : 0; }
            gsc[wave][lane] = (lane < groups && g == g && rank < keep) ? 1.0f : 0.0f;      // (a sum of two choice scores may be minus infinity with an expert left in the group)
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront"); __builtin_amdgcn_wave_barrier(); __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
#pragma unroll
            for (int i = 0; i < NV; i++) { const int e = lane + 64 * i; if (e < E && gsc[wave][e / per] == 0.0f) ok[i] = false; }
        }
        int rank[NV];
#pragma unroll
        for (int i = 0; i < NV; i++) { rank[i] = 0; if (!ok[i]) c[i] = -INFINITY; }
#pragma unroll
        for (int j = 0; j < NV; j++) {
#pragma unroll 16
            for (int l = 0; l < 64; l++) {
                const float o = __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(c[j]), l));
#pragma unroll
                for (int i = 0; i < NV; i++) rank[i] += (o > c[i] || (o == c[i] && l + 64 * j < lane + 64 * i)) ? 1 : 0;
            }
        }
        int chosen = 0;
#pragma unroll
        for (int i = 0; i < NV; i++) { if (!ok[i]) rank[i] = 1 << 20; chosen += __popcll(__ballot(rank[i] < top)); }
        float wsum = 0.0f;
        for (int r = 0; r < top; r++) {                      // in order of choice
            float w = 0.0f;
#pragma unroll
            for (int i = 0; i < NV; i++) {
                const unsigned long long m = __ballot(rank[i] == r);
                if (m) w = __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(s[i]), __ffsll(m) - 1));
            }
            wsum += w;
        }
        const float rinv = renorm ? 1.0f / (wsum + 1e-20f) : 1.0f;
        auto put = [&](int r, int e, float w) {
            ids[(size_t)t * top + r] = e; wts[(size_t)t * top + r] = w;
            if (SORT) { s_ids[wave * top + r] = e; s_w[wave * top + r] = w; }
        };
#pragma unroll
        for (int i = 0; i < NV; i++) if (rank[i] < top) put(rank[i], lane + 64 * i, renorm ? s[i] * rinv : s[i]);
        for (int r = chosen + lane; r < top; r += 64) put(r, 0, renorm ? 0.0f * rinv : 0.0f);      // fewer allowed experts than `top` (refused on the host): zero-weight slots
    }
    if (!SORT) return;
    __syncthreads();
    const int n = T * top;
    for (int i = threadIdx.x; i < n; i += 1024) atomicAdd(&cnt[s_ids[i]], 1);
    __syncthreads();
    if (wave == 0) {                                         // starts of the experts' rows: a prefix sum over two counters per lane
        const int a = cnt[2 * lane], b = cnt[2 * lane + 1];
        int sum = a + b;
#pragma unroll
        for (int o = 1; o < 64; o <<= 1) { const int v = __shfl_up(sum, o); if (lane >= o) sum += v; }
        const int at = sum - a - b;
        if (2 * lane < E) seg[2 * lane] = at;
        if (2 * lane + 1 < E) seg[2 * lane + 1] = at + a;
        if (lane == 63) seg[E] = sum;
        cnt[2 * lane] = at; cnt[2 * lane + 1] = at + a;
    }
    __syncthreads();
    for (int i = threadIdx.x; i < n; i += 1024) {
        const int e = s_ids[i], pos = atomicAdd(&cnt[e], 1);
        src_row[pos] = i / top; row_group[pos] = e; pair_pos[i] = pos;
        if (row_w) row_w[pos] = s_w[i];
    }
}
template <int NV, bool SORT>
__global__ void __launch_bounds__(SORT ? 1024 : 256) sv_router_rank_kernel(const KrSvRoute ro) { sv_router_rank<NV, SORT>(ro, blockIdx.x); }

// A parallel block's router reads the same product as its queries and keys: at decode sizes one launch does both, workgroup 0 the choice and the sort, the others sixteen
// (token, head) rows each.  A launch that depends on the one before it costs 4 - 5 us here whatever it does: one request 4.7 + 4.7 us as two launches, now 5.2.
template <int NV>
__global__ void __launch_bounds__(1024) sv_prep_route_kernel(const KrSvAttn a, const KrSvRoute ro, int heads_per_token) {
    extern __shared__ float hv16[];          // [16][dim]
    if (blockIdx.x == 0) { sv_router_rank<NV, true>(ro, 0); return; }
    const int wave = threadIdx.x >> 6, i = (blockIdx.x - 1) * 16 + wave;
    if (i < a.T * heads_per_token) sv_qk_prep_row<uint16_t>(a, i / heads_per_token, i % heads_per_token, threadIdx.x & 63, hv16 + wave * a.dim);
}

// Rows of a prompt's pairs sorted by expert, without atomics on a few hot words of memory (64 counters for 24576 pairs: 39 us to count and 39 us to place): a block counts its
// SORT_PAIRS pairs in LDS, one workgroup turns the blocks' counts into their first rows, the blocks place their pairs from LDS cursors (three launches of 5 us).
constexpr int SORT_PAIRS = 2048;
__global__ void __launch_bounds__(256) sv_moe_count_kernel(const int* __restrict__ ids, int n, int E, int* __restrict__ hist) {
    extern __shared__ int cnt[];             // [E]
    for (int e = threadIdx.x; e < E; e += 256) cnt[e] = 0;
    __syncthreads();
    const int i1 = min(n, (blockIdx.x + 1) * SORT_PAIRS);
    for (int i = blockIdx.x * SORT_PAIRS + threadIdx.x; i < i1; i += 256) atomicAdd(&cnt[ids[i]], 1);
    __syncthreads();
    for (int e = threadIdx.x; e < E; e += 256) hist[(size_t)blockIdx.x * E + e] = cnt[e];
}
__global__ void __launch_bounds__(1024) sv_moe_scan_kernel(int* __restrict__ hist, int blocks, int E, int* __restrict__ seg) {
    __shared__ int wsum[16]; __shared__ int carry;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    if (threadIdx.x == 0) carry = 0;
    for (int e0 = 0; e0 < E; e0 += 1024) {
        const int e = e0 + threadIdx.x;
        int tot = 0;
        if (e < E) for (int b = 0; b < blocks; b++) tot += hist[(size_t)b * E + e];
        int sum = tot;
#pragma unroll
        for (int o = 1; o < 64; o <<= 1) { const int v = __shfl_up(sum, o); if (lane >= o) sum += v; }
        __syncthreads();
        if (lane == 63) wsum[wave] = sum;
        __syncthreads();
        int at = carry + sum - tot;
        for (int w = 0; w < wave; w++) at += wsum[w];
        if (e < E) {
            seg[e] = at;
            for (int b = 0; b < blocks; b++) { const size_t i = (size_t)b * E + e; const int c = hist[i]; hist[i] = at; at += c; }
            if (e == E - 1) seg[E] = at;
        }
        __syncthreads();
        if (threadIdx.x == 1023) { int c = carry; for (int w = 0; w < 16; w++) c += wsum[w]; carry = c; }
        __syncthreads();
    }
}
__global__ void __launch_bounds__(256) sv_moe_fill_kernel(const int* __restrict__ ids, int n, int top, int E, const int* __restrict__ hist, int* __restrict__ src_row,
                                                          int* __restrict__ row_group, int* __restrict__ pair_pos, const float* __restrict__ wts, float* __restrict__ row_w) {
    extern __shared__ int cnt[];             // [E] next row of this block's pairs of the expert
    for (int e = threadIdx.x; e < E; e += 256) cnt[e] = hist[(size_t)blockIdx.x * E + e];
    __syncthreads();
    const int i1 = min(n, (blockIdx.x + 1) * SORT_PAIRS);
    for (int i = blockIdx.x * SORT_PAIRS + threadIdx.x; i < i1; i += 256) {
        const int e = ids[i];
        const int pos = atomicAdd(&cnt[e], 1);
        src_row[pos] = i / top; row_group[pos] = e; pair_pos[i] = pos;
        if (row_w) row_w[pos] = wts[i];
    }
}

// the same as one workgroup, for decode-sized batches (n pairs <= 1024)
__global__ void __launch_bounds__(256) sv_moe_sort_small_kernel(const int* __restrict__ ids, int n, int top, int E, int* __restrict__ seg, int* __restrict__ src_row,
                                                                int* __restrict__ row_group, int* __restrict__ pair_pos, const float* __restrict__ wts, float* __restrict__ row_w) {
    extern __shared__ int cnt[];             // [E] counts, then the next row of the expert
    for (int e = threadIdx.x; e < E; e += 256) cnt[e] = 0;
    __syncthreads();
    for (int i = threadIdx.x; i < n; i += 256) atomicAdd(&cnt[ids[i]], 1);
    __syncthreads();
    if (threadIdx.x < 64) {                  // 64 experts at a time through a prefix sum over the lanes
        int o = 0;
        for (int e0 = 0; e0 < E; e0 += 64) {
            const int e = e0 + (int)threadIdx.x, c = e < E ? cnt[e] : 0;
            int sum = c;
#pragma unroll
            for (int d = 1; d < 64; d <<= 1) { const int v = __shfl_up(sum, d); if ((int)threadIdx.x >= d) sum += v; }
            if (e < E) { seg[e] = o + sum - c; cnt[e] = o + sum - c; }
            o += __shfl(sum, 63);
        }
        if (threadIdx.x == 0) seg[E] = o;
    }
    __syncthreads();
    for (int i = threadIdx.x; i < n; i += 256) {
        const int e = ids[i];
        const int pos = atomicAdd(&cnt[e], 1);
        src_row[pos] = i / top; row_group[pos] = e; pair_pos[i] = pos;
        if (row_w) row_w[pos] = wts[i];
    }
}

template <typename T>
__global__ void sv_act_kernel(const float* __restrict__ gu, int ld, T* __restrict__ y, int M, int F, int kind, float limit, float alpha,
                              const float* __restrict__ row_w, const T* __restrict__ up_tab, const int* __restrict__ up_rows, int up_ld, int up_off) {
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= (size_t)M * F) return;
    const size_t r = i / F; const int c = (int)(i - r * F);
    float g = gu[r * ld + c], u = kind == KR_SV_ACT_RELU2 ? 0.0f : up_tab ? sv_ld(up_tab + (size_t)up_rows[r] * up_ld + up_off + c) : gu[r * ld + F + c];
    if (row_w) { g *= row_w[r]; u *= row_w[r]; }
    sv_st(y + i, gm_act_once(g, u, kind, limit, alpha));
}

// one workgroup per token: the sublayers' output row is formed in LDS, normed there when the design norms sublayer outputs, gated when the design gates
// them, added to the residual row, and the new row is written back and handed on in the storage type -- normed for the next sublayer (norm_w) or as it is
// NT threads: 256 for prompt-sized steps (many rows), 1024 for decode-sized ones, where a row's workgroup is alone on its compute unit and the
// per-thread chain of columns is what the launch waits for
template <typename T, int KIND, int NT>
__global__ void __launch_bounds__(NT) sv_residual_norm_kernel(const KrSvResidual a, T* __restrict__ h_out) {
    extern __shared__ float xr[];            // [width] | [2 * groups]
    __shared__ float red[NT / 64];
    __shared__ int pp_s[64]; __shared__ float w_s[64];      // the token's expert rows and weights, read once (top <= 64; more fall back to global reads)
    const size_t t = blockIdx.x;
    const int width = a.width, top = a.top;
    float* gst = xr + width;
    const float* __restrict__ rows = a.rows; const float* __restrict__ mix = a.mix; const float* __restrict__ dense = a.dense; const float* __restrict__ shared = a.shared;
    float* __restrict__ x = a.x;
    if (a.canon_state) {                     // the mixer's un-convolved input of this token is kept when it is among the last canon_keep of its portion
        const int K = a.canon_keep, sl = a.slot[t];
        if ((int)t + K >= a.T || a.slot[t + K] != sl) {
            float* dst = a.canon_state + ((size_t)sl * K + a.pos[t] % K) * width;
            for (int c = threadIdx.x; c < width; c += NT) dst[c] = a.h32_in[t * width + c];
        }
    }
    const bool staged = rows && top <= 64;
    if (staged && threadIdx.x < top) { pp_s[threadIdx.x] = a.pair_pos[t * top + threadIdx.x]; w_s[threadIdx.x] = a.wts ? a.wts[t * top + threadIdx.x] : 1.0f; }
    if (rows) __syncthreads();
    auto gate_at = [&](int c) {
        const float z = a.gate[t * a.ld_gate + c] + (a.gate_b ? a.gate_b[c] : 0.0f);
        return 1.0f / (1.0f + expf(-z));
    };
    float s1 = 0.0f;
    for (int c = threadIdx.x; c < width; c += NT) {
        const size_t i = t * width + c;
        float ff = 0.0f; bool any = false;
        if (rows) {
            if (staged) {
#pragma unroll 4
                for (int s = 0; s < top; s++) ff = __builtin_fmaf(w_s[s], rows[(size_t)pp_s[s] * width + c], ff);
            } else {
                for (int s = 0; s < top; s++) ff = __builtin_fmaf(a.wts ? a.wts[t * top + s] : 1.0f, rows[(size_t)a.pair_pos[t * top + s] * width + c], ff);
            }
            any = true;
        }
        if (shared) { ff = any ? ff + shared[i] : shared[i]; any = true; }
        if (dense) { ff = any ? ff + dense[i] : dense[i]; any = true; }
        float d = mix ? mix[i] : 0.0f;
        if (mix && a.mix_bias) d += a.mix_bias[c];
        if (any) d = mix ? d + ff : ff;
        if (a.post_w) { xr[c] = d; s1 += d; continue; }      // the sum waits for its norm
        if (a.gate) d *= gate_at(c);
        const float v = x[i] + a.mult * d;
        x[i] = v; xr[c] = v; s1 += v;
    }
    if (a.post_w) {
        float mean = 0.0f, inv = 0.0f;
        if (a.groups > 1) { __syncthreads(); sv_group_stats<KIND, NT / 64>(xr, width, a.groups, a.eps, gst); __syncthreads(); }
        else {
            if constexpr (KIND == KR_SV_NORM_LAYER) mean = sv_block_sum<NT / 64>(s1, red) / (float)width;
            float q = 0.0f;
            for (int c = threadIdx.x; c < width; c += NT) { const float dv = xr[c] - mean; q = __builtin_fmaf(dv, dv, q); }
            inv = 1.0f / sqrtf(sv_block_sum<NT / 64>(q, red) / (float)width + a.eps);
        }
        const int gw = a.groups > 1 ? width / a.groups : width;
        s1 = 0.0f;
        for (int c = threadIdx.x; c < width; c += NT) {
            const size_t i = t * width + c;
            if (a.groups > 1) { mean = gst[2 * (c / gw)]; inv = gst[2 * (c / gw) + 1]; }
            float y = (xr[c] - mean) * inv * a.post_w[c];
            if (a.post_b) y += a.post_b[c];
            if (a.gate) y *= gate_at(c);
            const float v = x[i] + a.mult * y;
            x[i] = v; xr[c] = v; s1 += v;
        }
    }
    if (!h_out) return;
    if (!a.norm_w) {
        for (int c = threadIdx.x; c < width; c += NT) { sv_st(h_out + t * width + c, xr[c]); if (a.h32_out) a.h32_out[t * width + c] = xr[c]; }
        return;
    }
    float mean = 0.0f, inv = 0.0f;
    if (a.groups > 1) { __syncthreads(); sv_group_stats<KIND, NT / 64>(xr, width, a.groups, a.eps, gst); __syncthreads(); }
    else {
        if constexpr (KIND == KR_SV_NORM_LAYER) mean = sv_block_sum<NT / 64>(s1, red) / (float)width;
        float q = 0.0f;
        for (int c = threadIdx.x; c < width; c += NT) { const float dv = xr[c] - mean; q = __builtin_fmaf(dv, dv, q); }      // a thread re-reads its own columns
        inv = 1.0f / sqrtf(sv_block_sum<NT / 64>(q, red) / (float)width + a.eps);
    }
    const int gw = a.groups > 1 ? width / a.groups : width;
    for (int c = threadIdx.x; c < width; c += NT) {
        if (a.groups > 1) { mean = gst[2 * (c / gw)]; inv = gst[2 * (c / gw) + 1]; }
        float v = (xr[c] - mean) * inv * a.norm_w[c];
        if (a.norm_b) v += a.norm_b[c];
        sv_st(h_out + t * width + c, v);
        if (a.h32_out) a.h32_out[t * width + c] = v;
    }
}

// the residual row in registers (see the row kernels above); an expert row's weight and place are the same for the whole workgroup (scalar loads), NB of them are requested together
template <typename T, int KIND, int NT, int CH>
__global__ void __launch_bounds__(NT) sv_residual_vec_kernel(const KrSvResidual a, T* __restrict__ h_out) {
    constexpr int NB = CH <= 2 ? 8 : 4;
    __shared__ float red[NT / 64];
    extern __shared__ __attribute__((aligned(16))) float row[];
    const size_t t = blockIdx.x;
    const int width = a.width, top = a.top;
    const size_t base = t * width;
    if (a.canon_state) {                     // the mixer's un-convolved input of this token is kept when it is among the last canon_keep of its portion
        const int K = a.canon_keep, sl = a.slot[t];
        if ((int)t + K >= a.T || a.slot[t + K] != sl) {
            float* dst = a.canon_state + ((size_t)sl * K + a.pos[t] % K) * width;
#pragma unroll
            for (int j = 0; j < CH; j++) { const int c = 4 * (threadIdx.x + NT * j); if (c < width) sv_st4(dst + c, sv_ld4(a.h32_in + base + c)); }
        }
    }
    float4 x[CH], d[CH];
    const float4 zero = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    auto add = [](float4 p, float4 q) { return make_float4(p.x + q.x, p.y + q.y, p.z + q.z, p.w + q.w); };
#pragma unroll
    for (int j = 0; j < CH; j++) { const int c = 4 * (threadIdx.x + NT * j); d[j] = zero; x[j] = c < width ? sv_ld4(a.x + base + c) : zero; }
    const bool any = a.rows || a.shared || a.dense;
    if (a.rows) {
        for (int s0 = 0; s0 < top; s0 += NB) {
            float4 r[NB][CH]; float w[NB];
#pragma unroll
            for (int u = 0; u < NB; u++) {
                if (s0 + u >= top) continue;
                const float* src = a.rows + (size_t)a.pair_pos[t * top + s0 + u] * width;
                w[u] = a.wts ? a.wts[t * top + s0 + u] : 1.0f;
#pragma unroll
                for (int j = 0; j < CH; j++) { const int c = 4 * (threadIdx.x + NT * j); r[u][j] = c < width ? sv_ld4(src + c) : zero; }
            }
#pragma unroll
            for (int u = 0; u < NB; u++) {
                if (s0 + u >= top) continue;
#pragma unroll
                for (int j = 0; j < CH; j++) {
                    d[j].x = __builtin_fmaf(w[u], r[u][j].x, d[j].x); d[j].y = __builtin_fmaf(w[u], r[u][j].y, d[j].y);
                    d[j].z = __builtin_fmaf(w[u], r[u][j].z, d[j].z); d[j].w = __builtin_fmaf(w[u], r[u][j].w, d[j].w);
                }
            }
        }
    }
    auto gated = [&](float4 v, int c) {
        float y[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
        for (int e = 0; e < 4; e++) { const float z = a.gate[t * a.ld_gate + c + e] + (a.gate_b ? a.gate_b[c + e] : 0.0f); y[e] *= 1.0f / (1.0f + expf(-z)); }
        return make_float4(y[0], y[1], y[2], y[3]);
    };
    auto joined = [&](float4 p, float4 q) { return make_float4(p.x + a.mult * q.x, p.y + a.mult * q.y, p.z + a.mult * q.z, p.w + a.mult * q.w); };
#pragma unroll
    for (int j = 0; j < CH; j++) {
        const int c = 4 * (threadIdx.x + NT * j);
        if (c >= width) continue;
        if (a.shared) d[j] = a.rows ? add(d[j], sv_ld4(a.shared + base + c)) : sv_ld4(a.shared + base + c);
        if (a.dense) d[j] = (a.rows || a.shared) ? add(d[j], sv_ld4(a.dense + base + c)) : sv_ld4(a.dense + base + c);
        if (a.mix) {
            float4 m = sv_ld4(a.mix + base + c);
            if (a.mix_bias) m = add(m, sv_ld4(a.mix_bias + c));
            d[j] = any ? add(m, d[j]) : m;
        }
    }
    if (a.post_w) sv_row_norm<KIND, NT, CH>(d, width, a.groups, a.eps, a.post_w, a.post_b, red, row);      // the sum passes its norm first
#pragma unroll
    for (int j = 0; j < CH; j++) {
        const int c = 4 * (threadIdx.x + NT * j);
        if (c >= width) continue;
        x[j] = joined(x[j], a.gate ? gated(d[j], c) : d[j]);
        sv_st4(a.x + base + c, x[j]);
    }
    if (!h_out) return;
    if (a.norm_w) sv_row_norm<KIND, NT, CH>(x, width, a.groups, a.eps, a.norm_w, a.norm_b, red, row);
#pragma unroll
    for (int j = 0; j < CH; j++) {
        const int c = 4 * (threadIdx.x + NT * j);
        if (c < width) { sv_st4(h_out + base + c, x[j]); if (a.h32_out) sv_st4(a.h32_out + base + c, x[j]); }
    }
}

// ---- latent mixer
// the rotated part of a key or query: thread `tid` of `nt` turns its pairs of z [rot] into dst
template <typename T>
__device__ __forceinline__ void sv_latent_turn(const float* z, const float2* cs, int rot, int interleaved, T* dst, int tid, int nt) {
    const int half = rot / 2;
    for (int i = tid; i < half; i += nt) {
        const int i0 = interleaved ? 2 * i : i, i1 = interleaved ? 2 * i + 1 : i + half;
        const float u = z[i0], v = z[i1];
        const float2 c = cs[i];
        sv_st(dst + i0, u * c.x - v * c.y); sv_st(dst + i1, v * c.x + u * c.y);
    }
}
// dst = z / rms(z) * w over n elements, by a workgroup of 256
template <typename T>
__device__ __forceinline__ void sv_latent_rms(const float* z, const float* w, int n, float eps, T* dst, float* red) {
    float q = 0.0f;
    for (int c = threadIdx.x; c < n; c += 256) q = __builtin_fmaf(z[c], z[c], q);
    const float inv = 1.0f / sqrtf(sv_block_sum<4>(q, red) / (float)n + eps);
    for (int c = threadIdx.x; c < n; c += 256) sv_st(dst + c, z[c] * inv * w[c]);
}
// the cache row of token t: [normed latent | turned shared key part]
template <typename T>
__device__ __forceinline__ void sv_latent_kv_row(const KrSvLatent& a, int t, int off, float* red) {
    const float* z = a.dz + (size_t)t * a.ld + off;
    const int p = a.pos[t];
    const size_t page = (size_t)a.page_table[(size_t)a.slot[t] * a.table_ld + p / a.page_tokens];
    T* dst = (T*)a.pool + (page * a.page_tokens + (p % a.page_tokens)) * (size_t)(a.kv_rank + a.rot);
    sv_latent_rms(z, a.dkv_norm_w, a.kv_rank, a.eps, dst, red);
    sv_latent_turn(z + a.kv_rank, a.cs + (size_t)t * (a.rot / 2), a.rot, a.rot_interleaved, dst + a.kv_rank, threadIdx.x, 256);
}
// head h of token t, by one wave: the plain part in the storage type, the turned part into the latent-wide query
template <typename T>
__device__ __forceinline__ void sv_latent_q_head(const KrSvLatent& a, const float* q, int t, int h, T* qn, float* qe, int lane) {
    T* n = qn + ((size_t)t * a.heads + h) * a.dim;
    for (int d = lane; d < a.dim; d += 64) sv_st(n + d, q[d]);
    sv_latent_turn(q + a.dim, a.cs + (size_t)t * (a.rot / 2), a.rot, a.rot_interleaved, qe + ((size_t)t * a.heads + h) * (a.kv_rank + a.rot) + a.kv_rank, lane, 64);
}
// one workgroup per (token, part): part 0 norms the query latent, part 1 norms the key / value latent into the cache row and turns the shared key part
template <typename T>
__global__ void __launch_bounds__(256) sv_latent_prep_kernel(const KrSvLatent a) {
    __shared__ float red[4];
    const int t = blockIdx.x;
    if (blockIdx.y) sv_latent_kv_row<T>(a, t, a.q_rank, red);
    else sv_latent_rms(a.dz + (size_t)t * a.ld, a.dq_norm_w, a.q_rank, a.eps, (T*)a.cq + (size_t)t * a.q_rank, red);
}
// one wave per (token, head)
template <typename T>
__global__ void __launch_bounds__(64) sv_latent_q_kernel(const KrSvLatent a, const float* __restrict__ q2, T* __restrict__ qn, float* __restrict__ qe) {
    const int t = blockIdx.x, h = blockIdx.y;
    sv_latent_q_head(a, q2 + ((size_t)t * a.heads + h) * (a.dim + a.rot), t, h, qn, qe, threadIdx.x);
}
// queries without a latent of their own: parts 0 .. ceil(heads / 4) - 1 take four heads each, a wave per head; the last part (own_kv) writes the cache row
template <typename T>
__global__ void __launch_bounds__(256) sv_latent_direct_kernel(const KrSvLatent a, T* __restrict__ qn, float* __restrict__ qe) {
    __shared__ float red[4];
    const int t = blockIdx.x, n = a.heads * (a.dim + a.rot);
    if ((int)blockIdx.y == (a.heads + 3) / 4) { sv_latent_kv_row<T>(a, t, n, red); return; }
    const int h = blockIdx.y * 4 + (threadIdx.x >> 6);
    if (h < a.heads) sv_latent_q_head(a, a.dz + (size_t)t * a.ld + (size_t)h * (a.dim + a.rot), t, h, qn, qe, threadIdx.x & 63);
}
__global__ void sv_head_rows_kernel(int T, int heads, int* __restrict__ seg, int* __restrict__ rows, int* __restrict__ group) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i <= heads) seg[i] = i * T;
    if (i >= T * heads) return;
    const int h = i / T, t = i - h * T;
    rows[i] = t * heads + h; group[i] = h;
}

// ---- recurrent mixers (KrSvLin)
// One WAVE per (request of the step, head, block of 16 value columns): lane = 4 * column + part, and a lane keeps the rows [part * dpr, (part + 1) * dpr) of
// its column of S in registers for the whole portion (dpr = ceil(dim / 4) <= DP).  The tokens of the portion are walked in order; TB of them at a time are
// staged in LDS (q and k of the head with the rotation and the scales applied, the 16 value columns, the two gates), so the serial loop reads LDS only.
// Per token a lane does dpr updates S <- a S + (b v) k and dpr products for o, and the four parts of a column meet through two lane exchanges.
#define SV_WAVE_SYNC() do { __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront"); __builtin_amdgcn_wave_barrier(); __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront"); } while (0)
template <int KIND, int DP>
__global__ void __launch_bounds__(64) sv_lin_scan_kernel(const KrSvLin a) {
    extern __shared__ __attribute__((aligned(16))) float lds[];
    constexpr int TB = 8;
    constexpr bool ML = KIND == 3, GLA = KIND == 4, SSD = KIND == 5, WKV = KIND == 7, DELTA = KIND == 8;
    const int e = blockIdx.x, h = blockIdx.y, cb = blockIdx.z, lane = threadIdx.x;
    const int part = lane & 3, cl = lane >> 2, col = cb * 16 + cl;
    const int dim = a.dim, vdim = a.vdim, H = a.heads, ncb = (vdim + 15) / 16;
    const int dpr = (dim + 3) / 4, dimp = 4 * dpr;
    const int t0 = a.ent_off[e], t1 = a.ent_off[e + 1], sl = a.ent_slot[e];
    const bool fresh = a.pos[t0] == 0, cv = col < vdim;
    float* Sg = a.state + (size_t)sl * a.state_stride + ((size_t)h * vdim + (cv ? col : 0)) * dim + part * dpr;
    float* nmg = a.nm + (size_t)sl * a.nm_stride + ((size_t)h * ncb + cb) * (dim + 4);
    float S[DP], n[DP];
#pragma unroll
    for (int r = 0; r < DP; r++) {
        const int row = part * dpr + r;
        const bool ok = r < dpr && row < dim && !fresh;
        S[r] = (ok && cv) ? Sg[r] : 0.0f;
        n[r] = (ML && ok) ? nmg[row] : 0.0f;
    }
    float m = (ML && !fresh) ? nmg[dim] : 0.0f;
    const float decay = KIND == 2 ? a.decay[h] : 0.0f;
    float* qs = lds; float* ks = qs + TB * dimp; float* vs = ks + TB * dimp; float* gs = vs + TB * 16; float* as = gs + TB * 2;      // as [TB * dimp]: per-channel decays (gla, wkv)
    float* us = as + TB * dimp;              // [dimp]: the current token's bonus (wkv)
    if constexpr (WKV) for (int d = lane; d < dimp; d += 64) us[d] = d < dim ? a.bonus[(size_t)h * dim + d] : 0.0f;
    const int half = a.rot_dims / 2;
    for (int tb = t0; tb < t1; tb += TB) {
        const int nt = min(TB, t1 - tb);
        if constexpr (GLA || SSD || WKV || DELTA) {
            const int hq = h / a.qk_group;
            for (int idx = lane; idx < nt * dimp; idx += 64) {
                const int tt = idx / dimp, d = idx - tt * dimp;
                const size_t r = (size_t)(tb + tt) * a.src_ld + (size_t)hq * dim + d;
                qs[idx] = d < dim ? a.qsrc[r] * a.q_scale : 0.0f;
                ks[idx] = d < dim ? a.ksrc[r] * a.k_scale : 0.0f;
                if constexpr (GLA) {
                    float al = 0.0f;
                    if (d < dim) {
                        const float z = a.gz[(size_t)(tb + tt) * a.gz_ld + (size_t)h * dim + d] + a.gz_bias[(size_t)h * dim + d];
                        al = expf((fminf(z, 0.0f) - log1pf(expf(-fabsf(z)))) * a.inv_tau);      // sigmoid(z)^(1 / tau)
                    }
                    as[idx] = al;
                }
                if constexpr (WKV) as[idx] = d < dim ? expf(a.gz[(size_t)(tb + tt) * a.gz_ld + (size_t)h * dim + d]) : 0.0f;
            }
            for (int idx = lane; idx < nt * 16; idx += 64) {
                const int tt = idx >> 4, c = cb * 16 + (idx & 15);
                vs[idx] = c < vdim ? a.vsrc[(size_t)(tb + tt) * a.src_ld + (size_t)h * vdim + c] : 0.0f;
            }
            if (SSD && lane < nt) {
                const float z = a.dtz[(size_t)(tb + lane) * a.dtz_ld + h] + a.dt_bias[h];
                const float dt = fmaxf(z, 0.0f) + log1pf(expf(-fabsf(z)));                      // softplus
                gs[2 * lane] = dt; gs[2 * lane + 1] = -expf(a.a_log[h]) * dt;
            }
            if (DELTA && lane < nt) { const float4 tk = a.tok[(size_t)(tb + lane) * H + h]; gs[2 * lane] = tk.w; gs[2 * lane + 1] = tk.x; }
        } else {
        for (int idx = lane; idx < nt * dimp; idx += 64) {
            const int tt = idx / dimp, d = idx - tt * dimp;
            const float* zr = a.z + (size_t)(tb + tt) * a.ld + (size_t)h * dim;
            qs[idx] = d < dim ? zr[d] * a.q_scale : 0.0f;
            ks[idx] = d < dim ? zr[(size_t)H * dim + d] * a.k_scale : 0.0f;
        }
        for (int idx = lane; idx < nt * 16; idx += 64) {
            const int tt = idx >> 4, c = cb * 16 + (idx & 15);
            vs[idx] = c < vdim ? a.z[(size_t)(tb + tt) * a.ld + (size_t)2 * H * dim + (size_t)h * vdim + c] : 0.0f;
        }
        if (ML && lane < nt) {
            const float* zg = a.z + (size_t)(tb + lane) * a.ld + (size_t)2 * H * dim + (size_t)2 * H * vdim;
            float zi = zg[h] + a.i_bias[h], zf = zg[H + h] + a.f_bias[h];
            if (a.gate_cap > 0.0f) { zi = a.gate_cap * tanhf(zi / a.gate_cap); zf = a.gate_cap * tanhf(zf / a.gate_cap); }
            gs[2 * lane] = zi;
            gs[2 * lane + 1] = fminf(zf, 0.0f) - log1pf(expf(-fabsf(zf)));      // log sigmoid
        }
        }
        SV_WAVE_SYNC();
        if (half > 0) {
            for (int idx = lane; idx < nt * half; idx += 64) {
                const int tt = idx / half, i = idx - tt * half;
                const float2 c = a.cs[(size_t)(tb + tt) * half + i];
                float* qp = qs + tt * dimp; float* kp = ks + tt * dimp;
                const float qu = qp[i], qv = qp[i + half], ku = kp[i], kv = kp[i + half];
                qp[i] = qu * c.x - qv * c.y; qp[i + half] = qv * c.x + qu * c.y;
                kp[i] = ku * c.x - kv * c.y; kp[i + half] = kv * c.x + ku * c.y;
            }
            SV_WAVE_SYNC();
        }
        for (int tt = 0; tt < nt; tt++) {
            const float* qp = qs + tt * dimp + part * dpr; const float* kp = ks + tt * dimp + part * dpr;
            const float v = vs[tt * 16 + cl];
            float av, bv;
            if constexpr (ML) {
                const float ig = gs[2 * tt], fg = gs[2 * tt + 1];
                const float mn = fmaxf(fg + m, ig);
                av = expf(fg + m - mn); bv = expf(ig - mn); m = mn;
            } else if constexpr (SSD || DELTA) { bv = gs[2 * tt]; av = expf(gs[2 * tt + 1]); }
            else { av = decay; bv = 1.0f; }
            const float* ap = as + tt * dimp + part * dpr; const float* up = us + part * dpr;
            float bvv = bv * v;
            float po = 0.0f, pn = 0.0f;
            if constexpr (DELTA) {                 // the decayed state's value at k first: what is written is the rest of v
                float pk = 0.0f;
#pragma unroll
                for (int r = 0; r < DP; r++) if (r < dpr) { S[r] *= av; pk = __builtin_fmaf(S[r], kp[r], pk); }
                pk += __shfl_xor(pk, 1); pk += __shfl_xor(pk, 2);
                bvv = bv * (v - pk); av = 1.0f;
            }
#pragma unroll
            for (int r = 0; r < DP; r++) {
                if (r < dpr) {
                    const float kr = kp[r], qr = qp[r];
                    if constexpr (WKV) {           // the read-out comes before the write
                        const float kv = kr * bvv;
                        po = __builtin_fmaf(__builtin_fmaf(up[r], kv, S[r]), qr, po);
                        S[r] = __builtin_fmaf(ap[r], S[r], kv);
                        continue;
                    }
                    if constexpr (GLA) S[r] = __builtin_fmaf(kr, bvv, ap[r] * S[r]);
                    else if constexpr (DELTA) S[r] = __builtin_fmaf(kr, bvv, S[r]);
                    else S[r] = __builtin_fmaf(kr, bvv, av * S[r]);
                    po = __builtin_fmaf(S[r], qr, po);
                    if constexpr (ML) { n[r] = __builtin_fmaf(bv, kr, av * n[r]); pn = __builtin_fmaf(n[r], qr, pn); }
                }
            }
            po += __shfl_xor(po, 1); po += __shfl_xor(po, 2);
            if constexpr (ML) {
                pn += __shfl_xor(pn, 1); pn += __shfl_xor(pn, 2);
                po = po / (fmaxf(fabsf(pn), expf(-m)) + 1e-6f);
            }
            if (part == 0 && cv) a.o[(size_t)(tb + tt) * H * vdim + (size_t)h * vdim + col] = po;
        }
        SV_WAVE_SYNC();
    }
#pragma unroll
    for (int r = 0; r < DP; r++) {
        const int row = part * dpr + r;
        if (r < dpr && row < dim) {
            if (cv) Sg[r] = S[r];
            if (ML && cl == 0) nmg[row] = n[r];
        }
    }
    if (ML && lane == 0) nmg[dim] = m;
}

// Prompt portions of the gla and state-space mixers (kinds 4, 5): the same recurrence, token by token, laid out for the length of the serial chain:
// what a portion waits for is the instructions ONE wave issues per token, so a head's state is spread over as many lanes as the chip has to spare.
// One WORKGROUP of four waves per (request, head, block of 8 value columns); a wave owns 2 columns, lane = 32 * column + part, and a lane keeps the rows
// [part * dpr, (part + 1) * dpr) of its column of S in registers (dpr = ceil(dim / 32) <= DP): a token costs a lane dpr updates and dpr products, and the
// thirty-two parts of a column meet in four exchanges inside their rows of 16 lanes and one across the two rows.  Tokens are staged 16 at a time in one
// of two LDS buffers: the loads of the next 16 are issued before the current 16 are walked and land in registers meanwhile (one barrier per 16
// tokens); the walk itself has no branch and no store (the 16 outputs of a lane leave together afterwards), so the LDS reads of the following tokens
// are in flight while one is worked on.  a.gz holds the decays themselves (sv_gla_decay_kernel).
// PIPE: the walk as an explicit pipeline (the next token's rows are read before the current one is worked on, the lane exchanges of all 16 tokens are done
// together afterwards) -- shorter when a workgroup has its compute unit to itself; with several workgroups per compute unit the plain walk (token after
// token, each with its own exchanges) leaves more of the issue slots to the others and the launch is over sooner.
template <int KIND, int DP, bool PIPE>
__global__ void __launch_bounds__(256) sv_lin_scanw_kernel(const KrSvLin a) {
    extern __shared__ __attribute__((aligned(16))) float lds[];
    constexpr int TB = 16, NC = 8;           // tokens per batch, value columns per workgroup
    constexpr bool GLA = KIND == 4, SSD = KIND == 5;
    const int e = blockIdx.x, h = blockIdx.y, cb = blockIdx.z, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int part = lane & 31, cl = wave * 2 + (lane >> 5), col = cb * NC + cl;
    const int dim = a.dim, vdim = a.vdim, H = a.heads;
    // a lane's dpr rows stand together in LDS, the parts of a token `pitch` floats apart: dpr + 4 where dpr is a multiple of 8, so that the 16-byte reads of
    // neighbouring parts fall into distinct banks
    const int dpr = (dim + 31) / 32, pitch = (dpr % 8 == 0) ? dpr + 4 : dpr, dimp = 32 * pitch;
    const int t0 = a.ent_off[e], t1 = a.ent_off[e + 1], sl = a.ent_slot[e];
    const bool fresh = a.pos[t0] == 0, cv = col < vdim;
    float* Sg = a.state + (size_t)sl * a.state_stride + ((size_t)h * vdim + (cv ? col : 0)) * dim + part * dpr;
    float S[DP];
#pragma unroll
    for (int r = 0; r < DP; r++) S[r] = (r < dpr && part * dpr + r < dim && !fresh && cv) ? Sg[r] : 0.0f;
    const int per = (GLA ? 3 : 2) * TB * dimp + TB * NC + TB * 2;      // floats of one buffer: q | k | (decays) | v | gates
    const int hq = h / a.qk_group;
    // staging: thread (token tid / 16 of the batch, row tid % 16 + 16 j of the head) -- 2 dpr elements of q, of k and of the decays per thread and batch.
    // fetch() is loads and nothing else (clamped addresses, no use of a loaded value), so that no wait stands between it and the walk over the current
    // batch; scales, masks and the gates' functions are applied when the registers go to LDS
    float pq[2 * DP], pk[2 * DP], pa[2 * DP], pv = 0.0f, pg = 0.0f;
    const int ft = tid >> 4, fd = tid & 15;
    int gd[2 * DP], li[2 * DP];              // per staged element: its column in the head's row (clamped) and its place in an LDS buffer
    unsigned real = 0;                       // bit j: the element exists (rows past dim are staged as zeros)
#pragma unroll
    for (int j = 0; j < 2 * DP; j++) {
        const int d = fd + 16 * j, pp = dpr == DP ? d / DP : d / dpr;
        gd[j] = min(d, dim - 1); li[j] = ft * dimp + pp * pitch + (d - pp * dpr);
        if (d < dim) real |= 1u << j;
    }
    auto fetch = [&](int tb) {               // global -> registers
        const int nt = min(TB, t1 - tb), tok = tb + min(ft, nt - 1);
        const size_t rb = (size_t)tok * a.src_ld + (size_t)hq * dim;
#pragma unroll
        for (int j = 0; j < 2 * DP; j++) {
            if (j < 2 * dpr) {
                const int d = gd[j];
                pq[j] = a.qsrc[rb + d]; pk[j] = a.ksrc[rb + d];
                if constexpr (GLA) pa[j] = a.gz[(size_t)tok * a.gz_ld + (size_t)h * dim + d];
            }
        }
        pv = a.vsrc[(size_t)(tb + min(tid >> 3, nt - 1)) * a.src_ld + (size_t)h * vdim + min(cb * NC + (tid & 7), vdim - 1)];      // threads below 128: (token, column)
        if constexpr (SSD) pg = a.dtz[(size_t)(tb + min(tid, nt - 1)) * a.dtz_ld + h];
    };
    const float ssd_rate = SSD ? -expf(a.a_log[h]) : 0.0f, ssd_bias = SSD ? a.dt_bias[h] : 0.0f;
    auto stash = [&](float* buf, int tb) {   // registers -> LDS
        const int nt = min(TB, t1 - tb);
        float* qs = buf; float* ks = qs + TB * dimp; float* as = ks + TB * dimp; float* vs = buf + (GLA ? 3 : 2) * TB * dimp; float* gs = vs + TB * NC;
#pragma unroll
        for (int j = 0; j < 2 * DP; j++)
            if (j < 2 * dpr) {
                const int idx = li[j];
                const bool ok = ft < nt && ((real >> j) & 1u);
                qs[idx] = ok ? pq[j] * a.q_scale : 0.0f; ks[idx] = ok ? pk[j] * a.k_scale : 0.0f;
                if constexpr (GLA) as[idx] = ok ? pa[j] : 0.0f;
            }
        if (tid < TB * NC) vs[tid] = ((tid >> 3) < nt && cb * NC + (tid & 7) < vdim) ? pv : 0.0f;
        if (SSD && tid < TB) {
            const float z = pg + ssd_bias;
            const float dt = fmaxf(z, 0.0f) + log1pf(expf(-fabsf(z)));      // softplus
            gs[2 * tid] = dt; gs[2 * tid + 1] = expf(ssd_rate * dt);
        }
    };
    fetch(t0); stash(lds, t0);
    __syncthreads();
    int b = 0;
    for (int tb = t0; tb < t1; tb += TB, b ^= 1) {
        const int nt = min(TB, t1 - tb);
        const bool more = tb + TB < t1;
        if (more) fetch(tb + TB);
        const float* buf = lds + b * per;
        const float* qs = buf; const float* ks = qs + TB * dimp; const float* as = ks + TB * dimp; const float* vs = buf + (GLA ? 3 : 2) * TB * dimp; const float* gs = vs + TB * NC;
        float outv[TB];
        if constexpr (PIPE) {
        // The walk, written as a pipeline: the lane's rows of q, k and the decays of token tt + 1 are read from LDS (16-byte reads when the lane's rows
        // fill DP) before token tt is worked on, and a token leaves only its lane's partial sum -- the exchanges among the 32 parts of a column are done
        // for all 16 tokens together afterwards, as 16 independent chains.  The state stays in registers; only S is carried from token to token.
        constexpr int G = 1;      // tokens read from LDS together, one group ahead of the group that is worked on
        float qq[2][G][DP], kk[2][G][DP], dd[2][G][DP], vv[2][G], g0[2][G], g1[2][G];      // two register sets, taken in turn (the loops are unrolled: every index is a constant)
        auto read = [&](int set, int t0g) {
            auto& qn = qq[set]; auto& kn = kk[set]; auto& dn = dd[set]; auto& vn = vv[set]; auto& g0n = g0[set]; auto& g1n = g1[set];
#pragma unroll
            for (int j = 0; j < G; j++) {
                const int tt = t0g + j;
                const float* qp = qs + tt * dimp + part * pitch; const float* kp = ks + tt * dimp + part * pitch; const float* ap = as + tt * dimp + part * pitch;
                if (dpr == DP) {
#pragma unroll
                    for (int r = 0; r < DP; r += 4) {
                        const float4 q4 = *reinterpret_cast<const float4*>(qp + r), k4 = *reinterpret_cast<const float4*>(kp + r);
                        qn[j][r] = q4.x; qn[j][r + 1] = q4.y; qn[j][r + 2] = q4.z; qn[j][r + 3] = q4.w; kn[j][r] = k4.x; kn[j][r + 1] = k4.y; kn[j][r + 2] = k4.z; kn[j][r + 3] = k4.w;
                        if constexpr (GLA) { const float4 a4 = *reinterpret_cast<const float4*>(ap + r); dn[j][r] = a4.x; dn[j][r + 1] = a4.y; dn[j][r + 2] = a4.z; dn[j][r + 3] = a4.w; }
                    }
                } else {
#pragma unroll
                    for (int r = 0; r < DP; r++) { qn[j][r] = r < dpr ? qp[r] : 0.0f; kn[j][r] = r < dpr ? kp[r] : 0.0f; if constexpr (GLA) dn[j][r] = r < dpr ? ap[r] : 0.0f; }
                }
                vn[j] = vs[tt * NC + cl];
                g0n[j] = SSD ? gs[2 * tt] : 1.0f; g1n[j] = SSD ? gs[2 * tt + 1] : 1.0f;
            }
        };
        read(0, 0);
        auto walk = [&](auto full) {             // full: all 16 tokens of the batch exist -- no branch anywhere in the walk
#pragma unroll
        for (int tg = 0; tg < TB; tg += G) {
            const int cur = (tg / G) & 1;
            if (tg + G < TB) read(cur ^ 1, tg + G);
            auto& qv = qq[cur]; auto& kv = kk[cur]; auto& dv = dd[cur];
            float av[G], bvv[G];
#pragma unroll
            for (int j = 0; j < G; j++) { av[j] = g1[cur][j]; bvv[j] = SSD ? vv[cur][j] * g0[cur][j] : vv[cur][j]; }
#pragma unroll
            for (int j = 0; j < G; j++) {
                const int tt = tg + j;
                float po0 = 0.0f, po1 = 0.0f;
                if (decltype(full)::value || tt < nt) {
#pragma unroll
                    for (int r = 0; r < DP; r += 2) {
                        if constexpr (GLA) { S[r] = __builtin_fmaf(kv[j][r], bvv[j], dv[j][r] * S[r]); S[r + 1] = __builtin_fmaf(kv[j][r + 1], bvv[j], dv[j][r + 1] * S[r + 1]); }
                        else { S[r] = __builtin_fmaf(kv[j][r], bvv[j], av[j] * S[r]); S[r + 1] = __builtin_fmaf(kv[j][r + 1], bvv[j], av[j] * S[r + 1]); }
                        po0 = __builtin_fmaf(S[r], qv[j][r], po0); po1 = __builtin_fmaf(S[r + 1], qv[j][r + 1], po1);
                    }
                }
                outv[tt] = po0 + po1;
            }
        }
        };
        if (nt == TB) walk(std::true_type{}); else walk(std::false_type{});
#pragma unroll
        for (int tt = 0; tt < TB; tt++) {
            float po = outv[tt];
            po += SV_DPPF(po, KR_DPP_XOR1); po += SV_DPPF(po, KR_DPP_XOR2); po += SV_DPPF(po, KR_DPP_HALF_MIRROR); po += SV_DPPF(po, KR_DPP_MIRROR);
            outv[tt] = po;
        }
#pragma unroll
        for (int tt = 0; tt < TB; tt++) outv[tt] += __shfl_xor(outv[tt], 16);
        } else {
        // one token: the lane's rows of q, k and the decays come from LDS (16-byte reads when the lane's rows fill DP), the state stays in registers
        auto token = [&](int tt) -> float {
            const float* qp = qs + tt * dimp + part * pitch; const float* kp = ks + tt * dimp + part * pitch; const float* ap = as + tt * dimp + part * pitch;
            float qv[DP], kv[DP], dv[DP];
            if (dpr == DP) {
#pragma unroll
                for (int r = 0; r < DP; r += 4) {
                    const float4 q4 = *reinterpret_cast<const float4*>(qp + r), k4 = *reinterpret_cast<const float4*>(kp + r);
                    qv[r] = q4.x; qv[r + 1] = q4.y; qv[r + 2] = q4.z; qv[r + 3] = q4.w; kv[r] = k4.x; kv[r + 1] = k4.y; kv[r + 2] = k4.z; kv[r + 3] = k4.w;
                    if constexpr (GLA) { const float4 a4 = *reinterpret_cast<const float4*>(ap + r); dv[r] = a4.x; dv[r + 1] = a4.y; dv[r + 2] = a4.z; dv[r + 3] = a4.w; }
                }
            } else {
#pragma unroll
                for (int r = 0; r < DP; r++) { qv[r] = r < dpr ? qp[r] : 0.0f; kv[r] = r < dpr ? kp[r] : 0.0f; if constexpr (GLA) dv[r] = r < dpr ? ap[r] : 0.0f; }
            }
            float av = 1.0f, bvv = vs[tt * NC + cl];
            if constexpr (SSD) { bvv *= gs[2 * tt]; av = gs[2 * tt + 1]; }
            float po0 = 0.0f, po1 = 0.0f;
#pragma unroll
            for (int r = 0; r < DP; r += 2) {
                if constexpr (GLA) { S[r] = __builtin_fmaf(kv[r], bvv, dv[r] * S[r]); S[r + 1] = __builtin_fmaf(kv[r + 1], bvv, dv[r + 1] * S[r + 1]); }
                else { S[r] = __builtin_fmaf(kv[r], bvv, av * S[r]); S[r + 1] = __builtin_fmaf(kv[r + 1], bvv, av * S[r + 1]); }
                po0 = __builtin_fmaf(S[r], qv[r], po0); po1 = __builtin_fmaf(S[r + 1], qv[r + 1], po1);
            }
            float po = po0 + po1;
            po += SV_DPPF(po, KR_DPP_XOR1); po += SV_DPPF(po, KR_DPP_XOR2); po += SV_DPPF(po, KR_DPP_HALF_MIRROR); po += SV_DPPF(po, KR_DPP_MIRROR);
            return po + __shfl_xor(po, 16);
        };
        if (nt == TB) {
#pragma unroll
            for (int tt = 0; tt < TB; tt++) outv[tt] = token(tt);
        } else {
#pragma unroll
            for (int tt = 0; tt < TB; tt++) outv[tt] = tt < nt ? token(tt) : 0.0f;
        }
        }
        if (more) stash(lds + (b ^ 1) * per, tb + TB);
        // the outputs leave after the registers of the next batch have gone to LDS: the wait for those loads then has no younger store before it
        if (part == 0 && cv) {
            float* op = a.o + (size_t)tb * H * vdim + (size_t)h * vdim + col;
#pragma unroll
            for (int tt = 0; tt < TB; tt++) if (tt < nt) op[(size_t)tt * H * vdim] = outv[tt];
        }
        __syncthreads();
    }
#pragma unroll
    for (int r = 0; r < DP; r++)
        if (r < dpr && part * dpr + r < dim && cv) Sg[r] = S[r];
}
// State-space mixer -> the block form of the recurrences: its recurrence is a retention whose decay changes from token to token,
// S_t = e^{l_t} S_(t-1) + (dt_t B_t) x_t^T with l_t = -e^{A_h} dt_t, read out by C_t.  One wave per (token, head) writes the head's own rows
// [q = C of its group | k = dt B of its group | v = x] where the block launches expect them and the token's log decay where sv_lin_prep_kernel would.
__global__ void __launch_bounds__(64) sv_ssd_expand_kernel(const KrSvLin a, float* __restrict__ zo, int ldz) {
    const int t = blockIdx.x, h = blockIdx.y, lane = threadIdx.x, H = a.heads, N = a.dim, dv = a.vdim, hq = h / a.qk_group;
    const float z = a.dtz[(size_t)t * a.dtz_ld + h] + a.dt_bias[h];
    const float dt = fmaxf(z, 0.0f) + log1pf(expf(-fabsf(z)));      // softplus
    const size_t r = (size_t)t * a.src_ld;
    float* o = zo + (size_t)t * ldz;
    for (int d = lane; d < N; d += 64) {
        o[(size_t)h * N + d] = a.qsrc[r + (size_t)hq * N + d];
        o[(size_t)H * N + (size_t)h * N + d] = a.ksrc[r + (size_t)hq * N + d] * dt;
    }
    for (int c = lane; c < dv; c += 64) o[(size_t)2 * H * N + (size_t)h * dv + c] = a.vsrc[r + (size_t)h * dv + c];
    if (lane == 0) a.tok[(size_t)t * H + h] = make_float4(-expf(a.a_log[h]) * dt, 0.0f, 0.0f, 0.0f);
}
// gla: the decays themselves from their logits, in place: a = sigmoid(z + b)^(1 / tau), formed through the logarithm
__global__ void sv_gla_decay_kernel(float* __restrict__ gz, const float* __restrict__ bias, size_t n, int cols, float inv_tau) {
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const float z = gz[i] + bias[i % cols];
    gz[i] = expf((fminf(z, 0.0f) - log1pf(expf(-fabsf(z)))) * inv_tau);
}

// ---- chunked form for prompt portions (KrSvLin: tok, sbuf, nbuf)
// rotation and scales on q / k in place, and the log gates of every (token, head): tok.x = log decay a, tok.y = log input b
__global__ void __launch_bounds__(64) sv_lin_prep_kernel(const KrSvLin a) {
    const int t = blockIdx.x, h = blockIdx.y, lane = threadIdx.x, H = a.heads, dim = a.dim;
    float* q = a.z + (size_t)t * a.ld + (size_t)h * dim; float* k = q + (size_t)H * dim;
    const int half = a.rot_dims / 2;
    for (int i = lane; i < half; i += 64) {
        const float2 c = a.cs[(size_t)t * half + i];
        const float qu = q[i] * a.q_scale, qv = q[i + half] * a.q_scale, ku = k[i] * a.k_scale, kv = k[i + half] * a.k_scale;
        q[i] = qu * c.x - qv * c.y; q[i + half] = qv * c.x + qu * c.y;
        k[i] = ku * c.x - kv * c.y; k[i + half] = kv * c.x + ku * c.y;
    }
    for (int d = a.rot_dims + lane; d < dim; d += 64) { q[d] *= a.q_scale; k[d] *= a.k_scale; }
    if (lane == 0) {
        float la, lb;
        if (a.kind == 3) {
            const float* zg = a.z + (size_t)t * a.ld + (size_t)2 * H * dim + (size_t)2 * H * a.vdim;
            float zi = zg[h] + a.i_bias[h], zf = zg[H + h] + a.f_bias[h];
            if (a.gate_cap > 0.0f) { zi = a.gate_cap * tanhf(zi / a.gate_cap); zf = a.gate_cap * tanhf(zf / a.gate_cap); }
            lb = zi; la = fminf(zf, 0.0f) - log1pf(expf(-fabsf(zf)));
        } else { la = fmaxf(logf(a.decay[h]), -1.0e4f); lb = 0.0f; }
        a.tok[(size_t)t * H + h] = make_float4(la, lb, 0.0f, 0.0f);
    }
}
// The running sum F of the log decays (from each block's start) and the running maximum m, m_t = F_t + max(m_start, max_(s <= t) (b_s - F_s)), in three
// launches: (1) a wave per (block, head) scans F and the prefix maximum of b - F over its 64 lanes, and leaves the block's last values; (2) a thread per
// (entry, head) carries m from block to block, m_next = F_last + max(m, pm_last), and leaves the last m in the slot's state; (3) a wave per (block, head)
// forms what the other launches read per token: (F - m, b - F, exp(F + m_start - m), exp(-m)).  Retention (b = 0, no maximum) is done after (1).
template <bool ML>
__global__ void __launch_bounds__(64) sv_lin_mlocal_kernel(const KrSvLin a) {
    const int gc = blockIdx.x, h = blockIdx.y, lane = threadIdx.x, H = a.heads;
    int e = 0;
    while (e + 1 < a.n_entries && a.ent_chunk0[e + 1] <= gc) e++;
    const int tb = a.ent_off[e] + 64 * (gc - a.ent_chunk0[e]), nt = min(64, a.ent_off[e + 1] - tb);
    const bool ok = lane < nt;
    const size_t ti = (size_t)(tb + lane) * H + h;
    float4 ab = make_float4(0.0f, -INFINITY, 0.0f, 0.0f);
    if (ok) { if (!ML && a.prepped == 2) ab.x = fmaxf(logf(a.decay[h]), -1.0e4f); else ab = a.tok[ti]; }
    float F = ab.x;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) { const float up = __shfl_up(F, o); if (lane >= o) F += up; }
    if constexpr (!ML) { if (ok) a.tok[ti] = make_float4(F, -F, expf(F), 0.0f); }
    else {
        const float x = ok ? ab.y - F : -INFINITY;
        float pm = x;
#pragma unroll
        for (int o = 1; o < 64; o <<= 1) { const float up = __shfl_up(pm, o); if (lane >= o) pm = fmaxf(pm, up); }
        if (ok) a.tok[ti] = make_float4(F, x, pm, 0.0f);
        if (lane == nt - 1) { float* cm = a.cmeta + ((size_t)gc * H + h) * 4; cm[0] = F; cm[1] = pm; }
    }
}
__global__ void __launch_bounds__(64) sv_lin_mchain_kernel(const KrSvLin a) {
    const int e = blockIdx.x, h = blockIdx.y * 64 + threadIdx.x, H = a.heads, ncb = (a.vdim + 15) / 16;
    if (h >= H) return;
    const int t0 = a.ent_off[e], nch = (a.ent_off[e + 1] - t0 + 63) / 64;
    float* nmh = a.nm + (size_t)a.ent_slot[e] * a.nm_stride + (size_t)h * ncb * (a.dim + 4);
    float m = a.pos[t0] != 0 ? nmh[a.dim] : 0.0f;
    float* cm = a.cmeta + ((size_t)a.ent_chunk0[e] * H + h) * 4; const size_t step = (size_t)H * 4;
    for (int c0 = 0; c0 < nch; c0 += 8) {                        // eight blocks' values are requested together: the chain itself is a few instructions a block
        float F[8], pm[8];
#pragma unroll
        for (int k = 0; k < 8; k++) { const size_t o = (size_t)min(c0 + k, nch - 1) * step; F[k] = cm[o]; pm[k] = cm[o + 1]; }
#pragma unroll
        for (int k = 0; k < 8; k++) if (c0 + k < nch) { cm[(size_t)(c0 + k) * step + 2] = m; m = F[k] + fmaxf(m, pm[k]); }
    }
    for (int cbk = 0; cbk < ncb; cbk++) nmh[(size_t)cbk * (a.dim + 4) + a.dim] = m;
}
__global__ void __launch_bounds__(64) sv_lin_mfinal_kernel(const KrSvLin a) {
    const int gc = blockIdx.x, h = blockIdx.y, lane = threadIdx.x, H = a.heads;
    int e = 0;
    while (e + 1 < a.n_entries && a.ent_chunk0[e + 1] <= gc) e++;
    const int tb = a.ent_off[e] + 64 * (gc - a.ent_chunk0[e]), nt = min(64, a.ent_off[e + 1] - tb);
    if (lane >= nt) return;
    const size_t ti = (size_t)(tb + lane) * H + h;
    const float m0 = a.cmeta[((size_t)gc * H + h) * 4 + 2];
    const float4 v = a.tok[ti];
    const float m = v.x + fmaxf(m0, v.z);
    a.tok[ti] = make_float4(v.x - m, v.y, expf(v.x + m0 - m), expf(-m));
}
// The state at every block's start, in two launches.  (1) In parallel over the blocks, one wave per (block, head, 16 value columns, NDT tiles of 16 key
// rows): the block's own contribution U = sum_s exp(u_last + w_s) k_s v_s^T on the matrix instruction (row d = 16 tile + 4 (lane / 16) + i, column =
// lane % 16), written where the block's start state will stand; the normaliser's contribution sum_s exp(u_last + w_s) k_s likewise.
template <bool ML, int NDT>
__global__ void __launch_bounds__(64) sv_lin_cupd_kernel(const KrSvLin a) {
    const int gcb = blockIdx.x, h = blockIdx.y, lane = threadIdx.x, r = lane & 15, kq = lane >> 4;
    const int H = a.heads, dim = a.dim, vdim = a.vdim, ncb = (vdim + 15) / 16;
    const int cb = blockIdx.z % ncb, dg = blockIdx.z / ncb;
    int e = 0;
    while (e + 1 < a.n_entries && a.ent_chunk0[e + 1] <= gcb) e++;
    const int tb = a.ent_off[e] + 64 * (gcb - a.ent_chunk0[e]), nt = min(64, a.ent_off[e + 1] - tb);
    const int col = cb * 16 + r; const bool cv = col < vdim;
    const float* zk = a.z + (size_t)H * dim + (size_t)h * dim; const float* zv = a.z + (size_t)2 * H * dim + (size_t)h * vdim;
    const float4 last = a.tok[(size_t)(tb + nt - 1) * H + h];
    float kk[16][NDT], vv[16], ww[16];
#pragma unroll
    for (int j = 0; j < 16; j++) {                                   // every operand of the block is requested before the first product
        const int s = 4 * j + kq; const size_t ts = (size_t)tb + min(s, nt - 1);
        ww[j] = s < nt ? a.tok[ts * H + h].y : -INFINITY;            // tokens past the portion's end weigh nothing
        vv[j] = cv ? zv[ts * a.ld + col] : 0.0f;
#pragma unroll
        for (int x = 0; x < NDT; x++) { const int da = (dg * NDT + x) * 16 + r; kk[j][x] = da < dim ? zk[ts * a.ld + da] : 0.0f; }
    }
    sv_f4 acc[NDT]; float nsum[NDT];
#pragma unroll
    for (int x = 0; x < NDT; x++) { acc[x] = sv_f4{0.0f, 0.0f, 0.0f, 0.0f}; nsum[x] = 0.0f; }
#pragma unroll
    for (int j = 0; j < 16; j++) {
        const float wgt = expf(last.x + ww[j]);
#pragma unroll
        for (int x = 0; x < NDT; x++) {
            const float aval = kk[j][x] * wgt;
            acc[x] = __builtin_amdgcn_mfma_f32_16x16x4f32(aval, vv[j], acc[x], 0, 0, 0);
            nsum[x] += aval;
        }
    }
    const size_t gc = (size_t)gcb * H + h;
#pragma unroll
    for (int x = 0; x < NDT; x++) {
        const int dt = dg * NDT + x;
#pragma unroll
        for (int i = 0; i < 4; i++) { const int d = dt * 16 + 4 * kq + i; if (cv && d < dim) a.sbuf[(gc * dim + d) * vdim + col] = acc[x][i]; }
        if constexpr (ML) {
            float v = nsum[x]; v += __shfl_xor(v, 16); v += __shfl_xor(v, 32);
            const int da = dt * 16 + r;
            if (cb == 0 && kq == 0 && da < dim) a.nbuf[gc * dim + da] = v;
        }
    }
}
// (2) Serial over the blocks of an entry, but element by element: a thread owns one element of S (or, in the last workgroups of a head, of the
// normaliser), walks the entry's blocks, leaves the state at the block's start where the block's contribution stood, and takes S <- g_last S + U.
// The contributions do not depend on the state, so their loads run ahead of the chain.
template <bool ML>
__global__ void __launch_bounds__(256) sv_lin_cscan_kernel(const KrSvLin a) {
    const int e = blockIdx.x, h = blockIdx.y, H = a.heads, dim = a.dim, vdim = a.vdim, ncb = (vdim + 15) / 16;
    const int t0 = a.ent_off[e], t1 = a.ent_off[e + 1], sl = a.ent_slot[e], c0 = a.ent_chunk0[e], nch = (t1 - t0 + 63) / 64;
    const bool fresh = a.pos[t0] == 0;
    const int idx = blockIdx.z * 256 + threadIdx.x;
    const int nS = dim * vdim;
    if (idx < nS) {
        const int d = idx / vdim, col = idx - d * vdim;
        float* Sg = a.state + (size_t)sl * a.state_stride + ((size_t)h * vdim + col) * dim + d;
        float S = fresh ? 0.0f : *Sg;
        float* p = a.sbuf + ((size_t)c0 * H + h) * nS + idx; const size_t step = (size_t)H * nS;
        int c = 0;
        for (; c + 4 <= nch; c += 4) {
            float u[4], g[4];
#pragma unroll
            for (int k = 0; k < 4; k++) { u[k] = p[(size_t)(c + k) * step]; g[k] = a.tok[(size_t)(min(t0 + 64 * (c + k + 1), t1) - 1) * H + h].z; }
#pragma unroll
            for (int k = 0; k < 4; k++) { p[(size_t)(c + k) * step] = S; S = __builtin_fmaf(g[k], S, u[k]); }
        }
        for (; c < nch; c++) {
            const float u = p[(size_t)c * step], g = a.tok[(size_t)(min(t0 + 64 * (c + 1), t1) - 1) * H + h].z;
            p[(size_t)c * step] = S; S = __builtin_fmaf(g, S, u);
        }
        *Sg = S;
    } else if (ML && idx - nS < dim) {
        const int d = idx - nS;
        float* nm = a.nm + (size_t)sl * a.nm_stride + (size_t)h * ncb * (dim + 4);
        float n = fresh ? 0.0f : nm[d];
        float* p = a.nbuf + ((size_t)c0 * H + h) * dim + d; const size_t step = (size_t)H * dim;
        for (int c = 0; c < nch; c++) {
            const float u = p[(size_t)c * step], g = a.tok[(size_t)(min(t0 + 64 * (c + 1), t1) - 1) * H + h].z;
            p[(size_t)c * step] = n; n = __builtin_fmaf(g, n, u);
        }
        for (int cbk = 0; cbk < ncb; cbk++) nm[(size_t)cbk * (dim + 4) + d] = n;      // every block of value columns keeps its own copy
    }
}
// parallel over blocks: a workgroup per (block, head), wave w owns the 16 tokens [16 w, 16 w + 16) of the block.  As in the matrix-instruction attention both
// products are formed transposed: S^T[s][t] = K Q^T (queries of the wave's tokens stay in registers: lane (t = lane % 16, quarter = lane / 16) keeps
// the quarter-th part of q_t), O^T[c][t] += V^T P^T with the weights where the first product left them; the state's share S_start^T q_t goes into the
// same accumulators first.  DQ >= ceil(dim / 4), DB >= ceil(vdim / 16).
// DIM > 0: that dim, vdim = 16 DB, key rows of whole 16-byte pieces (instances: 64 x 64, 64 x 128 and 128 x 128; other sizes, 128 x 64 among them, keep the guards); the queries in registers, so that four workgroups share a unit and not three.  A vector instruction between two f32 matrix instructions costs about 20 clocks (kr_serve_tile_f32.hip), and the
// guards put one beside every product: here products come in runs of 16 on operands read before them, from addresses that stand still.  Same products, same order.
// 3249 tokens of two requests, 16 heads of 128 x 128: 108 -> 55 us (three workgroups a unit 61; without the registers 91).
template <bool ML, int DB, int DIM>
__global__ void __launch_bounds__(256, DIM > 0 ? 4 : 1) sv_lin_cout_kernel(const KrSvLin a) {
    constexpr bool FULL = DIM > 0;
    constexpr int UNROLL = FULL ? DIM / 64 : 1;
    extern __shared__ __attribute__((aligned(16))) float sl[];      // [32][lds] rows of the block's start state | [4 waves][dq][64] the waves' queries
    const int gc = blockIdx.x, h = blockIdx.y, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, r = lane & 15, kq = lane >> 4;
    const int H = a.heads, dim = FULL ? DIM : a.dim, vdim = FULL ? 16 * DB : a.vdim, dq = 4 * ((dim + 15) / 16);
    const int lds = FULL ? 16 * DB + 16 : ((vdim + 31) / 32) * 32 + 16;      // rows 16 banks apart: the lanes of two neighbouring rows fall into distinct banks
    float* qs = sl + 32 * lds + (size_t)wave * dq * 64;             // this wave's queries, one word per (step, lane): a register file that loops can index
    int e = 0;
    while (e + 1 < a.n_entries && a.ent_chunk0[e + 1] <= gc) e++;
    const int tb = a.ent_off[e] + 64 * (gc - a.ent_chunk0[e]), nt = min(64, a.ent_off[e + 1] - tb);
    const bool active = wave * 16 < nt;                             // a wave without tokens still helps to stage the state
    const int trow = wave * 16 + r; const bool tv = trow < nt;
    const size_t tg = (size_t)tb + min(trow, nt - 1);
    const float4 me = a.tok[tg * H + h];
    const int grp = a.qk_group > 1 ? a.qk_group : 1, hq = h / grp, Hq = H / grp;      // heads of a group share one query and one key
    const float* zq = a.z + (size_t)hq * dim; const float* zk = zq + (size_t)Hq * dim; const float* zv = a.z + (size_t)2 * Hq * dim + (size_t)h * vdim;
    // the reduction index of a matrix instruction is spread over the four 16-lane groups: in step i lane group kq takes the key coordinate
    // d = 16 (i / 4) + 4 kq + i % 4, so that four steps of a lane are 16 contiguous bytes of a key row
    auto dof = [&](int i) { return 16 * (i >> 2) + 4 * kq + (i & 3); };
    const bool kvec = (a.ld & 3) == 0 && (dim & 15) == 0;          // key rows start 16-byte aligned and hold whole pieces
    float qr[FULL ? DIM / 4 : 1];
    if constexpr (FULL) {
#pragma unroll
        for (int j = 0; j < DIM / 16; j++) {
            const float4 q4 = *reinterpret_cast<const float4*>(zq + tg * a.ld + 16 * j + 4 * kq);
            qr[4 * j] = q4.x; qr[4 * j + 1] = q4.y; qr[4 * j + 2] = q4.z; qr[4 * j + 3] = q4.w;
        }
    } else
        for (int i = 0; i < dq; i++) { const int d = dof(i); qs[i * 64 + lane] = (active && d < dim) ? zq[tg * a.ld + d] : 0.0f; }
    sv_f4 acc[DB];
#pragma unroll
    for (int c = 0; c < DB; c++) acc[c] = sv_f4{0.0f, 0.0f, 0.0f, 0.0f};
    const float* Sc = a.sbuf + ((size_t)gc * H + h) * dim * vdim;
    const float* nc = a.nbuf + ((size_t)gc * H + h) * dim;
    float den = 0.0f;
    if constexpr (FULL) {
        constexpr int V4 = 4 * DB, NP = 32 * V4 / 256, G = 2;      // 16-byte pieces of a row; of a pass, per thread; steps whose rows are read together (four: 132 registers)
        sv_f4 pre[NP];
#pragma unroll
        for (int j = 0; j < NP; j++) pre[j] = reinterpret_cast<const sv_f4*>(Sc)[tid + 256 * j];
#pragma unroll
        for (int p0 = 0; p0 < DIM; p0 += 32) {
            __syncthreads();
#pragma unroll
            for (int j = 0; j < NP; j++) { const int idx = tid + 256 * j; *reinterpret_cast<sv_f4*>(sl + idx / V4 * lds + 4 * (idx % V4)) = pre[j]; }
            if (p0 + 32 < DIM) {
#pragma unroll
                for (int j = 0; j < NP; j++) pre[j] = reinterpret_cast<const sv_f4*>(Sc + (size_t)(p0 + 32) * vdim)[tid + 256 * j];
            }
            __syncthreads();
            if (active) {
            const float* srow = sl + 4 * kq * lds + r;
#pragma unroll
            for (int i4 = 0; i4 < 8; i4 += G) {
                float sv[G][DB];
#pragma unroll
                for (int i = 0; i < G; i++)
#pragma unroll
                    for (int c = 0; c < DB; c++) sv[i][c] = srow[(16 * ((i4 + i) >> 2) + ((i4 + i) & 3)) * lds + c * 16];
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int i = 0; i < G; i++)
#pragma unroll
                    for (int c = 0; c < DB; c++) acc[c] = __builtin_amdgcn_mfma_f32_16x16x4f32(sv[i][c], qr[p0 / 4 + i4 + i], acc[c], 0, 0, 0);
                if constexpr (ML) {
#pragma unroll
                    for (int i = 0; i < G; i++) den = __builtin_fmaf(qr[p0 / 4 + i4 + i], nc[p0 + dof(i4 + i)], den);
                }
                __builtin_amdgcn_sched_barrier(0);
            }
            }
        }
    } else
    for (int p0 = 0; p0 < dim; p0 += 32) {                          // passes over 32 rows of the state
        const int rows = min(32, dim - p0);
        __syncthreads();
        if ((vdim & 3) == 0) {                                      // 16-byte pieces: sbuf rows and the LDS rows are 16-byte aligned when vdim is a multiple of four
            const int v4 = vdim >> 2;
            for (int idx = tid; idx < rows * v4; idx += 256) {
                const int rr = idx / v4, c4 = idx - rr * v4;
                *reinterpret_cast<float4*>(sl + rr * lds + 4 * c4) = *reinterpret_cast<const float4*>(Sc + (size_t)(p0 + rr) * vdim + 4 * c4);
            }
        } else {
            for (int idx = tid; idx < rows * vdim; idx += 256) { const int rr = idx / vdim, cc = idx - rr * vdim; sl[rr * lds + cc] = Sc[(size_t)(p0 + rr) * vdim + cc]; }
        }
        __syncthreads();
        if (active) {
#pragma unroll 2
            for (int i = 0; i < 8; i++) {
                const int lr = dof(i);                            // row inside the pass (a pass is eight steps = 32 rows)
                const float qi = lr < rows ? qs[(p0 / 4 + i) * 64 + lane] : 0.0f;      // a row past dim meets a zero
                const float* srow = sl + min(lr, rows - 1) * lds + r;
#pragma unroll
                for (int c = 0; c < DB; c++) acc[c] = __builtin_amdgcn_mfma_f32_16x16x4f32(c * 16 + r < vdim ? srow[c * 16] : 0.0f, qi, acc[c], 0, 0, 0);
                if constexpr (ML) den = __builtin_fmaf(qi, nc[min(p0 + lr, dim - 1)], den);
            }
        }
    }
    if (!active) return;
    if constexpr (ML) { den += __shfl_xor(den, 16); den += __shfl_xor(den, 32); den *= me.z; }
#pragma unroll
    for (int c = 0; c < DB; c++) acc[c] *= me.z;
#pragma nounroll
    for (int stile = 0; stile <= wave; stile++) {
        const float* krow = zk + ((size_t)tb + min(stile * 16 + r, nt - 1)) * a.ld;
        sv_f4 st = sv_f4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll UNROLL
        for (int i0 = 0; i0 < dq; i0 += 16) {                    // sixteen key coordinates and queries requested at a time, then their products
            float kf[16], qf[16];
#pragma unroll
            for (int i = 0; i < 16; i++) qf[i] = FULL ? qr[FULL ? i0 + i : 0] : i0 + i < dq ? qs[(i0 + i) * 64 + lane] : 0.0f;
            if (FULL) {
#pragma unroll
                for (int j = 0; j < 4; j++) {
                    const float4 k4 = *reinterpret_cast<const float4*>(krow + 16 * (i0 / 4 + j) + 4 * kq);
                    kf[4 * j] = k4.x; kf[4 * j + 1] = k4.y; kf[4 * j + 2] = k4.z; kf[4 * j + 3] = k4.w;
                }
                __builtin_amdgcn_sched_barrier(0);
            } else if (kvec) {
#pragma unroll
                for (int j = 0; j < 4; j++) {
                    const float4 k4 = i0 + 4 * j < dq ? *reinterpret_cast<const float4*>(krow + 16 * (i0 / 4 + j) + 4 * kq) : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
                    kf[4 * j] = k4.x; kf[4 * j + 1] = k4.y; kf[4 * j + 2] = k4.z; kf[4 * j + 3] = k4.w;
                }
            } else {
#pragma unroll
                for (int i = 0; i < 16; i++) kf[i] = krow[min(dof(i0 + i), dim - 1)];
            }
#pragma unroll
            for (int i = 0; i < 16; i++) st = __builtin_amdgcn_mfma_f32_16x16x4f32(kf[i], qf[i], st, 0, 0, 0);
        }
        float ps = 0.0f;
        size_t srow[4];
#pragma unroll
        for (int i = 0; i < 4; i++) srow[i] = (size_t)tb + min(stile * 16 + 4 * kq + i, nt - 1);
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const int s = stile * 16 + 4 * kq + i;
            const bool ok = tv && s <= trow;
            const float p = ok ? st[i] * expf(me.x + a.tok[srow[i] * H + h].y) : 0.0f;
            st[i] = p; ps += p;
        }
        if constexpr (ML) { ps += __shfl_xor(ps, 16); ps += __shfl_xor(ps, 32); den += ps; }
        float vf[4][DB];                                          // the value rows of the tile's keys
#pragma unroll
        for (int i = 0; i < 4; i++)
#pragma unroll
            for (int c = 0; c < DB; c++) { const int cc = c * 16 + r; vf[i][c] = FULL || cc < vdim ? zv[srow[i] * a.ld + cc] : 0.0f; }
        if (FULL) __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int i = 0; i < 4; i++)
#pragma unroll
            for (int c = 0; c < DB; c++) acc[c] = __builtin_amdgcn_mfma_f32_16x16x4f32(vf[i][c], st[i], acc[c], 0, 0, 0);
        if (FULL) __builtin_amdgcn_sched_barrier(0);
    }
    const float inv = ML ? 1.0f / (fmaxf(fabsf(den), me.w) + 1e-6f) : 1.0f;
    if (!tv) return;
    float* o = a.o + tg * H * vdim + (size_t)h * vdim;
#pragma unroll
    for (int c = 0; c < DB; c++) {
        const int c0 = c * 16 + 4 * kq;
        if ((vdim & 3) == 0) { if (c0 < vdim) *reinterpret_cast<float4*>(o + c0) = make_float4(acc[c][0] * inv, acc[c][1] * inv, acc[c][2] * inv, acc[c][3] * inv); }
        else {
#pragma unroll
            for (int i = 0; i < 4; i++) if (c0 + i < vdim) o[c0 + i] = acc[c][i] * inv;
        }
    }
}

// one wave per (token, head): o / rms(o) (* weight) * act(g) -> the output projection's input
template <typename T>
__global__ void __launch_bounds__(64) sv_lin_out_kernel(const KrSvLin a, T* __restrict__ out) {
    const int t = blockIdx.x, h = blockIdx.y, lane = threadIdx.x, vdim = a.vdim, H = a.heads;
    const float* o = a.o + ((size_t)t * H + h) * vdim;
    const float* g = a.gate ? a.gate + (size_t)t * a.gate_ld + (size_t)h * vdim : a.z + (size_t)t * a.ld + (size_t)2 * H * a.dim + (size_t)H * vdim + (size_t)h * vdim;
    const bool sig = a.gate_act ? a.gate_act == 2 : a.kind == 3;
    float ss = 0.0f;
    for (int d = lane; d < vdim; d += 64) ss = __builtin_fmaf(o[d], o[d], ss);
    const float inv = 1.0f / sqrtf(sv_wave_sum(ss) / (float)vdim + a.eps);
    for (int d = lane; d < vdim; d += 64) {
        const float gz = g[d], sg = 1.0f / (1.0f + expf(-gz));
        float v = o[d] * inv;
        if (a.norm_w) v *= a.norm_w[a.norm_shared ? (size_t)d : (size_t)h * vdim + d];
        sv_st(out + ((size_t)t * H + h) * vdim + d, v * (sig ? sg : gz * sg));
    }
}

// A step that brings one token per request: scan and output of a head in ONE launch, a workgroup per (request, head) whose waves own 16 value columns each (lanes, registers and
// order of operations as in sv_lin_scan_kernel and sv_lin_out_kernel, so the bits are theirs).  What such a step waits for is not the state (64 KB per head at 128 x 128) but the
// trips to memory one after the other, and the second launch; here everything that does not hang on something read before (the state behind its slot, q, k, v, rotation, gates,
// norm) is requested first and waited for once.  dim = 4 DP rows exactly, so that a lane's rows are whole 16-byte pieces; other sizes stay with the two launches.
// 2 requests, 16 heads of 128 x 128: 12.2 + 4.6 -> 7.6 us.
template <int KIND, int DP>
__global__ void __launch_bounds__(512) sv_lin_step_kernel(const KrSvLin a, const bool f32) {
    constexpr bool ML = KIND == 3, GLA = KIND == 4, WKV = KIND == 7, DELTA = KIND == 8, SRC = GLA || WKV || DELTA;
    constexpr int dim = 4 * DP, PAD = DP + 4;              // the four parts of a column read LDS DP + 4 apart: no two in one bank
    __shared__ __attribute__((aligned(16))) float qs[4 * PAD], ks[4 * PAD], as[4 * PAD], us[4 * PAD], os[128];
    const int t = blockIdx.x, h = blockIdx.y, tid = threadIdx.x, lane = tid & 63, cb = tid >> 6, part = lane & 3, col = cb * 16 + (lane >> 2);
    const int vdim = a.vdim, H = a.heads, ncb = (vdim + 15) / 16, nt = blockDim.x, half = a.rot_dims / 2;
    const bool cv = col < vdim, fresh = a.pos[t] == 0;
    const int sl = a.ent_slot[t];
    float* Sg = a.state + (size_t)sl * a.state_stride + ((size_t)h * vdim + (cv ? col : 0)) * dim + part * DP;
    float* nmg = a.nm + (size_t)sl * a.nm_stride + ((size_t)h * ncb + cb) * (dim + 4);
    float4 S4[DP / 4], n4[DP / 4];
#pragma unroll
    for (int r = 0; r < DP / 4; r++) { S4[r] = *reinterpret_cast<const float4*>(Sg + 4 * r); if (ML) n4[r] = *reinterpret_cast<const float4*>(nmg + part * DP + 4 * r); }
    float m = ML ? nmg[dim] : 0.0f;
    const float* qp = SRC ? a.qsrc + (size_t)t * a.src_ld + (size_t)(h / a.qk_group) * dim : a.z + (size_t)t * a.ld + (size_t)h * dim;
    const float* kp = SRC ? a.ksrc + (size_t)t * a.src_ld + (size_t)(h / a.qk_group) * dim : qp + (size_t)H * dim;
    const float* vp = SRC ? a.vsrc + (size_t)t * a.src_ld + (size_t)h * vdim : a.z + (size_t)t * a.ld + (size_t)2 * H * dim + (size_t)h * vdim;
    const float* gp = a.gate ? a.gate + (size_t)t * a.gate_ld + (size_t)h * vdim : a.z + (size_t)t * a.ld + (size_t)2 * H * dim + (size_t)H * vdim + (size_t)h * vdim;
    const float v = cv ? vp[col] : 0.0f;
    const float gz = tid < vdim ? gp[tid] : 0.0f, nw = a.norm_w && tid < vdim ? a.norm_w[a.norm_shared ? (size_t)tid : (size_t)h * vdim + tid] : 1.0f;
    float av = 1.0f, bv = 1.0f;
    if constexpr (KIND == 2) av = a.decay[h];
    if constexpr (DELTA) { const float4 tk = a.tok[(size_t)t * H + h]; bv = tk.w; av = expf(tk.x); }
    if constexpr (ML) {
        const float* zg = a.z + (size_t)t * a.ld + (size_t)2 * H * dim + (size_t)2 * H * vdim;
        float zi = zg[h] + a.i_bias[h], zf = zg[H + h] + a.f_bias[h];
        if (a.gate_cap > 0.0f) { zi = a.gate_cap * tanhf(zi / a.gate_cap); zf = a.gate_cap * tanhf(zf / a.gate_cap); }
        const float fg = fminf(zf, 0.0f) - log1pf(expf(-fabsf(zf)));           // log sigmoid
        if (fresh) m = 0.0f;
        const float mn = fmaxf(fg + m, zi);
        av = expf(fg + m - mn); bv = expf(zi - mn); m = mn;
    }
    auto at = [](int d) { return d + 4 * (d / DP); };
    for (int i = tid; i < 2 * dim; i += nt) {              // q, then k; the thread of a rotated pair's first element turns both
        const int d = i & (dim - 1);
        const bool isk = i >= dim;
        const float* src = isk ? kp : qp;
        float* dst = isk ? ks : qs;
        const float sc = isk ? a.k_scale : a.q_scale;
        if (d < half) {
            const float2 c = a.cs[(size_t)t * half + d];
            const float u = src[d] * sc, w = src[d + half] * sc;
            dst[at(d)] = u * c.x - w * c.y; dst[at(d + half)] = w * c.x + u * c.y;
        } else if (d >= 2 * half) dst[at(d)] = src[d] * sc;
        if (!isk && GLA) {
            const float z = a.gz[(size_t)t * a.gz_ld + (size_t)h * dim + d] + a.gz_bias[(size_t)h * dim + d];
            as[at(d)] = expf((fminf(z, 0.0f) - log1pf(expf(-fabsf(z)))) * a.inv_tau);      // sigmoid(z)^(1 / tau)
        }
        if (!isk && WKV) { as[at(d)] = expf(a.gz[(size_t)t * a.gz_ld + (size_t)h * dim + d]); us[at(d)] = a.bonus[(size_t)h * dim + d]; }
    }
    __syncthreads();
    float bvv = bv * v, po = 0.0f, pn = 0.0f;
    const float *qr = qs + part * PAD, *kr = ks + part * PAD, *ar = as + part * PAD, *ur = us + part * PAD;
    float* S = reinterpret_cast<float*>(S4); float* n = reinterpret_cast<float*>(n4);
#pragma unroll
    for (int r = 0; r < DP; r++) { S[r] = fresh || !cv ? 0.0f : S[r]; if (ML) n[r] = fresh ? 0.0f : n[r]; }
    if constexpr (DELTA) {                                 // the decayed state's value at k first: what is written is the rest of v
        float pk = 0.0f;
#pragma unroll
        for (int r = 0; r < DP; r++) { S[r] *= av; pk = __builtin_fmaf(S[r], kr[r], pk); }
        pk += __shfl_xor(pk, 1); pk += __shfl_xor(pk, 2);
        bvv = bv * (v - pk);
    }
#pragma unroll
    for (int r = 0; r < DP; r++) {
        if constexpr (WKV) {                               // the read-out comes before the write
            const float kv = kr[r] * bvv;
            po = __builtin_fmaf(__builtin_fmaf(ur[r], kv, S[r]), qr[r], po);
            S[r] = __builtin_fmaf(ar[r], S[r], kv);
            continue;
        }
        if constexpr (GLA) S[r] = __builtin_fmaf(kr[r], bvv, ar[r] * S[r]);
        else if constexpr (DELTA) S[r] = __builtin_fmaf(kr[r], bvv, S[r]);
        else S[r] = __builtin_fmaf(kr[r], bvv, av * S[r]);
        po = __builtin_fmaf(S[r], qr[r], po);
        if constexpr (ML) { n[r] = __builtin_fmaf(bv, kr[r], av * n[r]); pn = __builtin_fmaf(n[r], qr[r], pn); }
    }
    po += __shfl_xor(po, 1); po += __shfl_xor(po, 2);
    if constexpr (ML) {
        pn += __shfl_xor(pn, 1); pn += __shfl_xor(pn, 2);
        po = po / (fmaxf(fabsf(pn), expf(-m)) + 1e-6f);
    }
    if (part == 0 && cv) os[col] = po;
#pragma unroll
    for (int r = 0; r < DP / 4; r++) {
        if (cv) *reinterpret_cast<float4*>(Sg + 4 * r) = S4[r];
        if (ML && (lane >> 2) == 0) *reinterpret_cast<float4*>(nmg + part * DP + 4 * r) = n4[r];
    }
    if (ML && lane == 0) nmg[dim] = m;
    __syncthreads();
    float ss = 0.0f;
    for (int d = lane; d < vdim; d += 64) ss = __builtin_fmaf(os[d], os[d], ss);
    const float inv = 1.0f / sqrtf(sv_wave_sum(ss) / (float)vdim + a.eps);
    if (tid < vdim) {
        const float sg = 1.0f / (1.0f + expf(-gz)), o = os[tid] * inv * nw;
        const bool sig = a.gate_act ? a.gate_act == 2 : ML;
        const size_t at_o = ((size_t)t * H + h) * vdim + tid;
        if (f32) ((float*)a.out)[at_o] = o * (sig ? sg : gz * sg); else sv_st((uint16_t*)a.out + at_o, o * (sig ? sg : gz * sg));
    }
}

// the selective state-space mixer after its scan (KrSvSsdOut): one workgroup per token, the gated row in LDS
template <typename T>
__global__ void __launch_bounds__(256) sv_ssd_out_kernel(const KrSvSsdOut a, T* __restrict__ out) {
    extern __shared__ float yr[];            // [inner] | [2 * groups]
    const size_t t = blockIdx.x;
    const int inner = a.heads * a.vdim;
    float* gst = yr + inner;
    for (int c = threadIdx.x; c < inner; c += 256) {
        const float xv = a.x[t * a.ld_x + c], zv = a.z[t * a.ld_z + c];
        yr[c] = __builtin_fmaf(a.D[c / a.vdim], xv, a.o[t * inner + c]) * (zv / (1.0f + expf(-zv)));
    }
    __syncthreads();
    sv_group_stats<KR_SV_NORM_RMS, 4>(yr, inner, a.groups, a.eps, gst);
    __syncthreads();
    const int gw = inner / a.groups;
    for (int c = threadIdx.x; c < inner; c += 256) sv_st(out + t * a.out_ld + c, yr[c] * gst[2 * (c / gw) + 1] * a.w[c] * a.scale);
}

// The end of a step, many workgroups per row: the row's largest entry (the lowest index of equals; NaN never), and the row itself, to pinned host memory.  Two copy commands and
// the host's wait for each took 40 us after this launch, 100 with 1.5 MB of logits; the stores here cross the link beside the search.
// best: value in order of size and index in one word, 0 = none yet; the last workgroup of a row hands the result on and leaves best and done as it found them.
__global__ void __launch_bounds__(256) sv_finish_kernel(const float* __restrict__ logits, int vocab, int chunk, float* const* host_logits, int* __restrict__ host_argmax,
                                                        unsigned long long* __restrict__ best, unsigned* __restrict__ done) {
    __shared__ unsigned long long bw[4];
    const int r = blockIdx.x, c0 = blockIdx.y * chunk, c1 = min(vocab, c0 + chunk);
    const float* row = logits + (size_t)r * vocab;
    float* to = gm_host(host_logits);
    if (to) to += (size_t)r * vocab;
    unsigned long long b = 0;
    auto see = [&](float x, int c) {
        if (x != x) return;
        const uint32_t u = __float_as_uint(x + 0.0f);          // (both zeros are equal)
        const unsigned long long k = ((unsigned long long)((u & 0x80000000u) ? ~u : u | 0x80000000u) << 32) | (0xFFFFFFFFu - (uint32_t)c);
        if (k > b) b = k;
    };
    if (vocab % 4 == 0) {
        for (int c = c0 + 4 * threadIdx.x; c < c1; c += 1024) {
            const float4 q = *reinterpret_cast<const float4*>(row + c);
            if (to) *reinterpret_cast<float4*>(to + c) = q;
            see(q.x, c); see(q.y, c + 1); see(q.z, c + 2); see(q.w, c + 3);
        }
    } else {
        for (int c = c0 + threadIdx.x; c < c1; c += 256) { const float x = row[c]; if (to) to[c] = x; see(x, c); }
    }
    if (!host_argmax) return;
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) { const unsigned long long v = __shfl_xor(b, o); if (v > b) b = v; }
    if ((threadIdx.x & 63) == 0) bw[threadIdx.x >> 6] = b;
    __syncthreads();
    if (threadIdx.x != 0) return;
    for (int w = 1; w < 4; w++) if (bw[w] > b) b = bw[w];
    __hip_atomic_fetch_max(best + r, b, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if (__hip_atomic_fetch_add(done + r, 1u, __ATOMIC_ACQ_REL, __HIP_MEMORY_SCOPE_AGENT) != gridDim.y - 1) return;
    const unsigned long long v = __hip_atomic_exchange(best + r, 0ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __hip_atomic_store(done + r, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    host_argmax[r] = v ? (int)(0xFFFFFFFFu - (uint32_t)v) : 0;
}
template <typename T>
__global__ void sv_fill_uniform_kernel(T* __restrict__ p, size_t n, uint64_t seed, float amp) {
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    uint64_t z = seed + 0x9E3779B97F4A7C15ull * (i + 1);      // splitmix64 of the element index
    z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull; z = (z ^ (z >> 27)) * 0x94D049BB133111EBull; z ^= z >> 31;
    const float u = (float)(z >> 40) * (1.0f / 16777216.0f);  // [0, 1)
    sv_st(p + i, (2.0f * u - 1.0f) * amp);
}
}  // namespace

void kr_sv_fill_uniform(void* p, bool f32, size_t n, uint64_t seed, float amp, hipStream_t st) {
    if (n == 0) return;
    const dim3 grid((unsigned)((n + 255) / 256));
    if (f32) hipLaunchKernelGGL(sv_fill_uniform_kernel<float>, grid, dim3(256), 0, st, (float*)p, n, seed, amp);
    else hipLaunchKernelGGL(sv_fill_uniform_kernel<uint16_t>, grid, dim3(256), 0, st, (uint16_t*)p, n, seed, amp);
}

void kr_sv_embed(const void* table, bool f32, const int* tokens, float* x, void* h_out, int T, int width, float scale, const void* table2, const int* rows2, hipStream_t st) {
    if (T <= 0) return;
    if (f32) hipLaunchKernelGGL(sv_embed_kernel<float>, dim3(T), dim3(256), 0, st, (const float*)table, tokens, x, (float*)h_out, width, scale, (const float*)table2, rows2);
    else hipLaunchKernelGGL(sv_embed_kernel<uint16_t>, dim3(T), dim3(256), 0, st, (const uint16_t*)table, tokens, x, (uint16_t*)h_out, width, scale, (const uint16_t*)table2, rows2);
}

void kr_sv_stream_norm(float* x, const float* add, const float* w, const float* b, bool in_place, void* out, bool out_f32, int T, int width, float eps, int kind, int groups,
                       hipStream_t st) {
    if (T <= 0 || (!add && !w)) return;
    const size_t lds = (size_t)(width + 2 * (groups > 1 ? groups : 0)) * sizeof(float);
#define SV_SN(T_, K_) hipLaunchKernelGGL((sv_stream_norm_kernel<T_, K_>), dim3(T), dim3(256), lds, st, x, add, w, b, (int)in_place, (T_*)out, width, eps, groups)
    if (kind == KR_SV_NORM_LAYER) { if (out_f32) SV_SN(float, KR_SV_NORM_LAYER); else SV_SN(uint16_t, KR_SV_NORM_LAYER); }
    else { if (out_f32) SV_SN(float, KR_SV_NORM_RMS); else SV_SN(uint16_t, KR_SV_NORM_RMS); }
#undef SV_SN
}

void kr_sv_chan_conv(const KrSvChanConv& c, hipStream_t st) {
    if (c.T <= 0 || c.C <= 0) return;
    hipLaunchKernelGGL(sv_chan_conv_kernel, dim3(c.T, (c.C + 255) / 256), dim3(256), 0, st, c);
}
void kr_sv_chan_conv_save(const KrSvChanConv& c, hipStream_t st) {
    if (c.T <= 0 || c.C <= 0 || c.taps < 2 || c.n_entries <= 0) return;
    hipLaunchKernelGGL(sv_chan_conv_save_kernel, dim3(c.n_entries, c.taps - 1, (c.C + 255) / 256), dim3(256), 0, st, c);
}
void kr_sv_scale(float* p, size_t n, float scale, hipStream_t st) {
    if (n == 0) return;
    hipLaunchKernelGGL(sv_scale_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, p, n, scale);
}
void kr_sv_ssd_out(const KrSvSsdOut& a, bool f32, hipStream_t st) {
    if (a.T <= 0) return;
    const size_t lds = (size_t)(a.heads * a.vdim + 2 * a.groups) * sizeof(float);
    if (f32) hipLaunchKernelGGL(sv_ssd_out_kernel<float>, dim3(a.T), dim3(256), lds, st, a, (float*)a.out);
    else hipLaunchKernelGGL(sv_ssd_out_kernel<uint16_t>, dim3(a.T), dim3(256), lds, st, a, (uint16_t*)a.out);
}

template <typename T, int KIND>
static void sv_norm_launch(const float* x, const int* rows, const float* w, const float* b, T* out, int R, int width, float eps, int groups, float* out32, hipStream_t st) {
    const size_t glds = groups > 1 ? (size_t)(width + 2 * groups) * sizeof(float) : 0;
    if (sv_al16({x, w, b, out, out32}) && sv_vec_rows(R, width, [&](auto nt, auto ch) {
            hipLaunchKernelGGL((sv_norm_vec_kernel<T, KIND, nt(), ch()>), dim3(R), dim3(nt()), glds, st, x, rows, w, b, out, width, eps, groups, out32); })) return;
    hipLaunchKernelGGL((sv_norm_kernel<T, KIND>), dim3(R), dim3(256), (size_t)2 * groups * sizeof(float), st, x, rows, w, b, out, width, eps, groups, out32);
}
void kr_sv_norm(const float* x, const int* rows, const float* w, const float* b, void* out, bool out_f32, int R, int width, float eps, int kind, int groups, float* out32,
                hipStream_t st) {
    if (R <= 0) return;
    if (kind == KR_SV_NORM_LAYER) { if (out_f32) sv_norm_launch<float, KR_SV_NORM_LAYER>(x, rows, w, b, (float*)out, R, width, eps, groups, out32, st); else sv_norm_launch<uint16_t, KR_SV_NORM_LAYER>(x, rows, w, b, (uint16_t*)out, R, width, eps, groups, out32, st); }
    else { if (out_f32) sv_norm_launch<float, KR_SV_NORM_RMS>(x, rows, w, b, (float*)out, R, width, eps, groups, out32, st); else sv_norm_launch<uint16_t, KR_SV_NORM_RMS>(x, rows, w, b, (uint16_t*)out, R, width, eps, groups, out32, st); }
}

template <typename T, int KIND>
static bool sv_embed_norm_launch(const T* table, const int* tokens, float* x, float scale, const T* table2, const int* rows2, const float* w, const float* b, T* out, int R, int width, float eps,
                                 int groups, float* out32, const KrSvBegin& bg, hipStream_t st) {
    const size_t glds = groups > 1 ? (size_t)(width + 2 * groups) * sizeof(float) : 0;
    return sv_al16({table, x, table2, w, b, out, out32}) && sv_vec_rows(R, width, [&](auto nt, auto ch) {
            hipLaunchKernelGGL((sv_embed_norm_kernel<T, KIND, nt(), ch()>), dim3(R + (bg.words > 0 ? sv_begin_blocks(bg, nt()) : 0)), dim3(nt()), glds, st, table, tokens, x, scale, table2, rows2, w, b,
                               out, width, eps, groups, out32, bg, R); });
}
bool kr_sv_embed_norm(const void* table, bool f32, const int* tokens, float* x, int T, int width, float scale, const void* table2, const int* rows2, const float* w, const float* b, void* out,
                      float eps, int kind, int groups, float* out32, const KrSvBegin& bg, hipStream_t st) {
    if (T <= 0) return true;
#define SV_ENL(T_, K_) sv_embed_norm_launch<T_, K_>((const T_*)table, tokens, x, scale, (const T_*)table2, rows2, w, b, (T_*)out, T, width, eps, groups, out32, bg, st)
    if (kind == KR_SV_NORM_LAYER) return f32 ? SV_ENL(float, KR_SV_NORM_LAYER) : SV_ENL(uint16_t, KR_SV_NORM_LAYER);
    return f32 ? SV_ENL(float, KR_SV_NORM_RMS) : SV_ENL(uint16_t, KR_SV_NORM_RMS);
#undef SV_ENL
}

void kr_sv_begin(const KrSvBegin& b, hipStream_t st) { hipLaunchKernelGGL(sv_begin_kernel, dim3(sv_begin_blocks(b, 256)), dim3(256), 0, st, b); }

void kr_sv_rope_table(const int* pos, const double* inv_freq, float2* cs, int T, int half, float mult, hipStream_t st) {
    const int n = T * half;
    if (n <= 0) return;
    hipLaunchKernelGGL(sv_rope_table_kernel, dim3((n + 255) / 256), dim3(256), 0, st, pos, inv_freq, cs, T, half, mult);
}

void kr_sv_qk_rms(const KrSvAttn& a, hipStream_t st) {
    if (a.T <= 0) return;
    hipLaunchKernelGGL(sv_qk_rms_kernel, dim3(a.T, 2), dim3(256), 0, st, a);
}

void kr_sv_canon(const KrSvCanon& c, bool f32, hipStream_t st) {
    if (c.T <= 0) return;
    const dim3 grid(c.T, (c.width + 255) / 256);
    if (f32) hipLaunchKernelGGL(sv_canon_kernel<float>, grid, dim3(256), 0, st, c, (float*)c.out);
    else hipLaunchKernelGGL(sv_canon_kernel<uint16_t>, grid, dim3(256), 0, st, c, (uint16_t*)c.out);
}

void kr_sv_qk_prep(const KrSvAttn& a, bool f32, hipStream_t st) {
    if (a.T <= 0) return;
    const dim3 grid(a.T, a.heads + (a.own_kv ? (a.v_from_k ? 1 : 2) * a.kv_heads : 0));
    const size_t lds = (size_t)a.dim * sizeof(float);
    if (f32) hipLaunchKernelGGL(sv_qk_prep_kernel<float>, grid, dim3(64), lds, st, a);
    else hipLaunchKernelGGL(sv_qk_prep_kernel<uint16_t>, grid, dim3(64), lds, st, a);
}

// the register tilings of the matrix-instruction attention: (dim / 4, vdim / 16)
static bool sv_mfma_tiling(int dq, int db) {
    static const int tab[][2] = {{16, 4}, {32, 8}, {16, 8}, {32, 4}, {8, 2}, {8, 4}, {16, 2}, {64, 16}, {64, 8}, {32, 16}, {8, 16}, {8, 1}, {16, 1},
                                 // latent cache rows: [latent | rotated part] as the key, the latent as the value (512 + 64, 256 + 64, 128 + 64 and the like)
                                 {144, 32}, {80, 16}, {48, 8}};
    for (const auto& t : tab) if (t[0] == dq && t[1] == db) return true;
    return false;
}
static bool sv_mfma_fits(int heads, int kv_heads, int dim, int vdim, int ldk, int ldv, bool f32) {
    const int VEC = f32 ? 4 : 8, R = heads / kv_heads;
    if (!((R <= 16 && 16 % R == 0) || R % 16 == 0)) return false;
    if (dim % (4 * VEC) != 0 || vdim % 16 != 0 || ldk % VEC != 0 || ldv % VEC != 0) return false;
    return sv_mfma_tiling(dim / 4, vdim / 16);
}
// keys a wave takes at a time in a split launch: long rows on the matrix path go 16 at a time (a wave's loads of one 64-key block are ~40 dependent
// batches at one wave per SIMD: a decode step is over sooner with four times the waves), everything else 64.  f32 rows of 128 elements are as long, up to 256 workgroups: a step of one
// layer, us, 64 -> 16 keys: one request at 250 / 500 / 2500 keys 207 / 207 / 212 -> 196 / 196 / 199, twelve at 300 608 -> 598, forty at 200 665 -> 635; but a portion of 250 tokens 564 -> 578.
static int sv_split_key_block(int T, int heads, int kv_heads, int dim, int vdim, int ldk, int ldv, bool f32) {
    const bool few = f32 && dim >= 128 && (long)T * kv_heads * ((heads / kv_heads + 15) / 16) <= 256;
    return (dim >= 192 || few) && sv_mfma_fits(heads, kv_heads, dim, vdim, ldk, ldv, f32) ? 16 : 64;
}

int kr_sv_attention_splits(int T, int heads, int kv_heads, int dim, int vdim, int ldk, int ldv, bool f32, int max_visible) {
    const int R = heads / kv_heads;
    const int vc = vdim <= 64 ? 1 : vdim <= 128 ? 2 : vdim <= 256 ? 4 : 8;
    const int rmax = vc <= 2 ? 16 : vc == 4 ? 8 : 4;
    int rm = 2;
    while (rm < R && rm < rmax) rm *= 2;
    const long blocks = (long)T * kv_heads * ((R + rm - 1) / rm);
    const int kblk = sv_split_key_block(T, heads, kv_heads, dim, vdim, ldk, ldv, f32);
    const int nch = (max_visible + kblk - 1) / kblk;
    long ns = 1024 / (blocks > 0 ? blocks : 1);              // about four workgroups per compute unit
    if (ns > (nch + 3) / 4) ns = (nch + 3) / 4;              // a workgroup keeps at least one block of keys per wave
    return ns < 1 ? 1 : (int)ns;
}

// Which form an entry of the step takes.  A single token goes to its own workgroups (per key head and 16 query heads), which read its keys for it alone; a portion of many tokens to
// 128-row tiles.  Portions of 2 - 31 tokens go either way: own workgroups while all short entries together are at most 192 of them, three quarters of the chip (us per step of two layers
// at 500 keys, own workgroups / tiles: 16 / 2 heads, one portion of 16 tokens 131 / 158, eight of 16 219 / 214, eight of 31 383 / 248; 8 / 8 heads, one of 8 143 / 158, one of 31 223 / 171;
// at 1500 keys, 64 portions of 16, 8 / 8 heads 3847 / 828, 64 / 4 heads 2888 / 1000).
// Short entries beside a prompt portion have rows in few waves of a tile and may see many more keys than the portion: they ride in its launch unless that makes them its tail by three
// tiles of keys or more, else they get a launch of their own before it (one request at 20000 keys beside 512 tokens, 64 / 4 heads: 3347 riding, 453 apart; beside 2000 tokens 3783 / 1125;
// but 15 requests at 200 keys beside 2000 tokens, 16 / 2 heads, window 1024: 522 / 563).
KrSvAttnPlan kr_sv_attn_form(int n_entries, const int* counts, const int* last_pos, int heads, int kv_heads, int dim, int vdim, int ldk, int ldv, int ldq, int page_tokens, bool f32, int window,
                             int keep, int chunk) {
    KrSvAttnPlan p{};
    const bool prompt = kr_sv_attn_prompt_fits(heads, kv_heads, dim, vdim, ldk, ldv, ldq, f32), step = kr_sv_attn_step_fits(dim, vdim, ldk, ldv, ldq, page_tokens, f32);
    struct Part { int tokens = 0, entries = 0, keys = 0; };      // of some entries: how many, and the most keys that one of their tokens sees
    auto part = [&](int lo, int hi) {
        Part q;
        for (int e = 0; e < n_entries; e++) {
            if (counts[e] < lo || counts[e] > hi) continue;
            const int n = last_pos[e] + 1;
            q.tokens += counts[e]; q.entries++;
            q.keys = std::max(q.keys, window > 0 ? std::min(n, window + keep) : chunk > 0 ? std::min(n, chunk) : n);
        }
        return q;
    };
    const Part all = part(1, INT_MAX), below = part(1, 31);
    p.keys = all.keys;
    // (where the tiles do not fit, no form shares a token's keys with the next token)
    const int few = !prompt || (long)below.tokens * kv_heads * ((heads / kv_heads + 15) / 16) <= 192 ? 31 : 1;
    const Part a = part(1, few), b = part(few + 1, INT_MAX);
    if (step && b.entries == 0) {
        p.form = KR_SV_ATTN_STEP; p.nsplit = kr_sv_attn_step_splits(all.tokens, heads, kv_heads, all.keys);
    } else if (prompt && (step || part(32, INT_MAX).entries > 0)) {      // (pages that own workgroups do not take: the general form up to 31 tokens)
        p.form = KR_SV_ATTN_PROMPT; p.nsplit = kr_sv_attn_prompt_splits(all.tokens, all.entries, heads, kv_heads, all.keys);
        if (step && a.entries > 0 && (a.keys + 63) / 64 - (b.keys + 63) / 64 >= 3 * p.nsplit) {
            p.few = few; p.n_few = a.tokens; p.nsplit_few = kr_sv_attn_step_splits(a.tokens, heads, kv_heads, a.keys);
            p.nsplit = kr_sv_attn_prompt_splits(b.tokens, b.entries, heads, kv_heads, b.keys);
        }
    } else {
        p.form = KR_SV_ATTN_GENERAL; p.nsplit = kr_sv_attention_splits(all.tokens, heads, kv_heads, dim, vdim, ldk, ldv, f32, all.keys);
    }
    p.parts = std::max(p.nsplit > 1 ? (size_t)all.tokens * p.nsplit : 0, p.nsplit_few > 1 ? (size_t)p.n_few * p.nsplit_few : 0) * heads;
    return p;
}

// the matrix-instruction form takes prompt-sized steps whose head sizes fit its register tiling
template <typename T>
static bool sv_attn_mfma_launch(const KrSvAttn& a, hipStream_t st) {
    if (!sv_mfma_fits(a.heads, a.kv_heads, a.dim, a.vdim, a.ldk, a.ldv, sizeof(T) == 4)) return false;
    const int R = a.heads / a.kv_heads;
    const int Rb = R < 16 ? R : 16;
    KrSvAttn b = a;
    b.tq = a.nsplit > 1 ? 1 : 16 / Rb;      // a split launch is a decode-shaped step: its tokens belong to different requests
    const dim3 grid((a.T + b.tq - 1) / b.tq, a.kv_heads, (R <= 16 ? 1 : R / 16) * a.nsplit);
    const size_t lds = (size_t)(4 * 16 * 2 + 16 * 2 + 16 * (a.vdim + 65)) * sizeof(float);
#define SV_MF(DQ_, DB_) do { hipLaunchKernelGGL((sv_attn_mfma_kernel<T, DQ_, DB_>), grid, dim3(256), lds, st, b); return true; } while (0)
#define SV_MF1(DQ_, DB_) do { if (a.nsplit > 1) hipLaunchKernelGGL((sv_attn_mfma_kernel<T, DQ_, DB_, 1>), grid, dim3(256), lds, st, b); \
                              else hipLaunchKernelGGL((sv_attn_mfma_kernel<T, DQ_, DB_>), grid, dim3(256), lds, st, b); return true; } while (0)
    const bool short_blocks = sv_split_key_block(a.T, a.heads, a.kv_heads, a.dim, a.vdim, a.ldk, a.ldv, sizeof(T) == 4) == 16;
#define SV_MF4(DQ_, DB_) do { if constexpr (sizeof(T) == 4) { if (short_blocks) SV_MF1(DQ_, DB_); } SV_MF(DQ_, DB_); } while (0)
    const int dq = a.dim / 4, db = a.vdim / 16;
    if (dq == 16 && db == 4) SV_MF(16, 4);
    if (dq == 32 && db == 8) SV_MF4(32, 8);
    if (dq == 16 && db == 8) SV_MF(16, 8);
    if (dq == 32 && db == 4) SV_MF4(32, 4);
    if (dq == 8 && db == 2) SV_MF(8, 2);
    if (dq == 8 && db == 4) SV_MF(8, 4);
    if (dq == 16 && db == 2) SV_MF(16, 2);
    if (dq == 64 && db == 16) SV_MF(64, 16);
    if (dq == 64 && db == 8) SV_MF(64, 8);
    if (dq == 32 && db == 16) SV_MF4(32, 16);
    if (dq == 8 && db == 16) SV_MF(8, 16);
    if (dq == 8 && db == 1) SV_MF(8, 1);
    if (dq == 16 && db == 1) SV_MF(16, 1);
    if (dq == 144 && db == 32) SV_MF1(144, 32);     // split launches of the long rows: 16 keys per wave at a time (sv_split_key_block)
    if (dq == 80 && db == 16) SV_MF1(80, 16);
    if (dq == 48 && db == 8) SV_MF1(48, 8);
#undef SV_MF
#undef SV_MF1
#undef SV_MF4
    return false;
}

void kr_sv_attn_merge(const KrSvAttn& a, hipStream_t st) {
    hipLaunchKernelGGL(sv_attn_merge_kernel<uint16_t>, dim3(a.T, a.heads), dim3(256), (size_t)(a.nsplit + 1) * sizeof(float), st, a);
}

void kr_sv_attention(const KrSvAttn& a, bool f32, hipStream_t st) {
    if (a.T <= 0) return;
    if (a.form != KR_SV_ATTN_GENERAL) {
        // the short entries' launches come first; both kinds leave partial states in the same buffers, one after the other
        KrSvAttn b = a;
        if (a.form == KR_SV_ATTN_PROMPT && a.n_few > 0) { b.form = KR_SV_ATTN_STEP; b.toks = a.order; b.T = a.n_few; b.nsplit = a.nsplit_few; }
        for (;;) {
            if (b.form == KR_SV_ATTN_PROMPT) kr_sv_attn_prompt(b, st); else kr_sv_attn_step(b, st);
            const int n = b.form == KR_SV_ATTN_PROMPT ? b.T - b.n_few : b.T;
            if (b.nsplit > 1) hipLaunchKernelGGL(sv_attn_merge_kernel<uint16_t>, dim3(n, b.heads), dim3(256), (size_t)(b.nsplit + 1) * sizeof(float), st, b);
            if (b.form == a.form) return;
            b = a; b.toks = a.order + a.n_few;
        }
    }
    if (f32 ? sv_attn_mfma_launch<float>(a, st) : sv_attn_mfma_launch<uint16_t>(a, st)) {
        if (a.nsplit > 1) {
            if (f32) hipLaunchKernelGGL(sv_attn_merge_kernel<float>, dim3(a.T, a.heads), dim3(256), (size_t)(a.nsplit + 1) * sizeof(float), st, a);
            else hipLaunchKernelGGL(sv_attn_merge_kernel<uint16_t>, dim3(a.T, a.heads), dim3(256), (size_t)(a.nsplit + 1) * sizeof(float), st, a);
        }
        return;
    }
    const int R = a.heads / a.kv_heads;
    const int vc = a.vdim <= 64 ? 1 : a.vdim <= 128 ? 2 : a.vdim <= 256 ? 4 : 8;
    const int rmax = vc <= 2 ? 16 : vc == 4 ? 8 : 4;       // RM * VC accumulators per lane stay within 32
    int rm = 2;
    while (rm < R && rm < rmax) rm *= 2;
    const dim3 grid(a.T, a.kv_heads, ((R + rm - 1) / rm) * a.nsplit);
    const size_t lds = ((size_t)rm * a.dim + 4 * 64 * rm + 8 * rm + (size_t)rm * a.vdim) * sizeof(float);
#define SV_ATT(T_, RM_, VC_) hipLaunchKernelGGL((sv_attn_group_kernel<T_, RM_, VC_>), grid, dim3(256), lds, st, a)
#define SV_ATT_R(T_, VC_) do { if (rm == 2) SV_ATT(T_, 2, VC_); else if (rm == 4) SV_ATT(T_, 4, VC_); else if (rm == 8) SV_ATT(T_, 8, VC_); else SV_ATT(T_, 16, VC_); } while (0)
#define SV_ATT_T(T_) do { if (vc == 1) SV_ATT_R(T_, 1); else if (vc == 2) SV_ATT_R(T_, 2); else if (vc == 4) { if (rm == 2) SV_ATT(T_, 2, 4); else if (rm == 4) SV_ATT(T_, 4, 4); else SV_ATT(T_, 8, 4); } \
                          else { if (rm == 2) SV_ATT(T_, 2, 8); else SV_ATT(T_, 4, 8); } } while (0)
    if (f32) SV_ATT_T(float); else SV_ATT_T(uint16_t);
    if (a.nsplit > 1) {
        if (f32) hipLaunchKernelGGL(sv_attn_merge_kernel<float>, dim3(a.T, a.heads), dim3(256), (size_t)(a.nsplit + 1) * sizeof(float), st, a);
        else hipLaunchKernelGGL(sv_attn_merge_kernel<uint16_t>, dim3(a.T, a.heads), dim3(256), (size_t)(a.nsplit + 1) * sizeof(float), st, a);
    }
#undef SV_ATT_T
#undef SV_ATT_R
#undef SV_ATT
}

size_t kr_sv_moe_hist_ints(int pairs, int E) { return pairs <= 1024 && E <= 4096 ? 0 : ((size_t)pairs + SORT_PAIRS - 1) / SORT_PAIRS * E; }

static bool sv_route_ranked(const KrSvRoute& r) { return r.E <= 128 && r.top <= 64 && r.groups <= 64; }

void kr_sv_router_sort(const KrSvRoute& r, int* hist, hipStream_t st) {
    const int T = r.T, E = r.E, top = r.top, groups = r.groups, n = T * top;
    int *ids = r.ids, *seg = r.seg, *src_row = r.src_row, *row_group = r.row_group, *pair_pos = r.pair_pos; float *wts = r.wts, *row_w = r.row_w;
    if (n <= 0) return;
    if (sv_route_ranked(r) && T <= 16) {                 // a wave per token, the sort in the same launch
        if (E <= 64) hipLaunchKernelGGL((sv_router_rank_kernel<1, true>), dim3(1), dim3(1024), 0, st, r);
        else hipLaunchKernelGGL((sv_router_rank_kernel<2, true>), dim3(1), dim3(1024), 0, st, r);
        return;
    }
    if (sv_route_ranked(r)) {
        if (E <= 64) hipLaunchKernelGGL((sv_router_rank_kernel<1, false>), dim3((T + 3) / 4), dim3(256), 0, st, r);
        else hipLaunchKernelGGL((sv_router_rank_kernel<2, false>), dim3((T + 3) / 4), dim3(256), 0, st, r);
    } else hipLaunchKernelGGL(sv_router_select_kernel, dim3(T), dim3(64), (size_t)(2 * E + 2 * groups) * sizeof(float), st, r.z, r.ld, r.parts, r.bias, r.bias_mode, r.score_kind, r.group_kind, E, top,
                              groups, r.keep, r.renorm, ids, wts);
    if (n <= 1024 && E <= 4096) {
        hipLaunchKernelGGL(sv_moe_sort_small_kernel, dim3(1), dim3(256), (size_t)E * sizeof(int), st, ids, n, top, E, seg, src_row, row_group, pair_pos, wts, row_w);
        return;
    }
    const int blocks = (n + SORT_PAIRS - 1) / SORT_PAIRS;
    hipLaunchKernelGGL(sv_moe_count_kernel, dim3(blocks), dim3(256), (size_t)E * sizeof(int), st, ids, n, E, hist);
    hipLaunchKernelGGL(sv_moe_scan_kernel, dim3(1), dim3(1024), 0, st, hist, blocks, E, seg);
    hipLaunchKernelGGL(sv_moe_fill_kernel, dim3(blocks), dim3(256), (size_t)E * sizeof(int), st, ids, n, top, E, hist, src_row, row_group, pair_pos, wts, row_w);
}

void kr_sv_prep_route(const KrSvAttn& a, const KrSvRoute& r, hipStream_t st) {
    const int hpt = a.heads + (a.own_kv ? (a.v_from_k ? 1 : 2) * a.kv_heads : 0);
    const size_t lds = (size_t)16 * a.dim * sizeof(float);
    const dim3 grid(1 + (a.T * hpt + 15) / 16), nt(1024);
    if (r.E <= 64) hipLaunchKernelGGL(sv_prep_route_kernel<1>, grid, nt, lds, st, a, r, hpt);
    else hipLaunchKernelGGL(sv_prep_route_kernel<2>, grid, nt, lds, st, a, r, hpt);
}

void kr_sv_act(const float* gu, int ld, void* y, bool f32, int M, int F, int kind, float limit, float alpha, const float* row_w, hipStream_t st, const void* up_tab,
               const int* up_rows, int up_ld, int up_off) {
    const size_t n = (size_t)M * F;
    if (n == 0) return;
    const dim3 grid((unsigned)((n + 255) / 256));
    if (f32) hipLaunchKernelGGL(sv_act_kernel<float>, grid, dim3(256), 0, st, gu, ld, (float*)y, M, F, kind, limit, alpha, row_w, (const float*)up_tab, up_rows, up_ld, up_off);
    else hipLaunchKernelGGL(sv_act_kernel<uint16_t>, grid, dim3(256), 0, st, gu, ld, (uint16_t*)y, M, F, kind, limit, alpha, row_w, (const uint16_t*)up_tab, up_rows, up_ld, up_off);
}

static bool sv_residual_al16(const KrSvResidual& r) {
    return sv_al16({r.x, r.mix, r.mix_bias, r.rows, r.shared, r.dense, r.post_w, r.post_b, r.norm_w, r.norm_b, r.h_out, r.h32_in, r.h32_out, r.canon_state});
}
bool kr_sv_residual_vec(const KrSvResidual& r) { return sv_residual_al16(r) && sv_vec_rows(r.T, r.width, [](auto, auto) {}); }
template <typename T, int KIND> static void sv_residual_launch(const KrSvResidual& r, hipStream_t st) {
    const size_t lds = (size_t)(r.width + 2 * (r.groups > 1 ? r.groups : 0)) * sizeof(float), glds = r.groups > 1 ? lds : 0;
    if (sv_residual_al16(r) &&
        sv_vec_rows(r.T, r.width, [&](auto nt, auto ch) { hipLaunchKernelGGL((sv_residual_vec_kernel<T, KIND, nt(), ch()>), dim3(r.T), dim3(nt()), glds, st, r, (T*)r.h_out); })) return;
    if (r.T <= 64) hipLaunchKernelGGL((sv_residual_norm_kernel<T, KIND, 1024>), dim3(r.T), dim3(1024), lds, st, r, (T*)r.h_out);
    else hipLaunchKernelGGL((sv_residual_norm_kernel<T, KIND, 256>), dim3(r.T), dim3(256), lds, st, r, (T*)r.h_out);
}
void kr_sv_residual_norm(const KrSvResidual& r, bool out_f32, hipStream_t st) {
    if (r.T <= 0) return;
    if (r.kind == KR_SV_NORM_LAYER) { if (out_f32) sv_residual_launch<float, KR_SV_NORM_LAYER>(r, st); else sv_residual_launch<uint16_t, KR_SV_NORM_LAYER>(r, st); }
    else { if (out_f32) sv_residual_launch<float, KR_SV_NORM_RMS>(r, st); else sv_residual_launch<uint16_t, KR_SV_NORM_RMS>(r, st); }
}

void kr_sv_latent_prep(const KrSvLatent& a, bool f32, hipStream_t st) {
    if (a.T <= 0) return;
    if (f32) hipLaunchKernelGGL(sv_latent_prep_kernel<float>, dim3(a.T, 2), dim3(256), 0, st, a);
    else hipLaunchKernelGGL(sv_latent_prep_kernel<uint16_t>, dim3(a.T, 2), dim3(256), 0, st, a);
}
void kr_sv_latent_q(const KrSvLatent& a, const float* q2, void* qn, float* qe, bool f32, hipStream_t st) {
    if (a.T <= 0) return;
    if (f32) hipLaunchKernelGGL(sv_latent_q_kernel<float>, dim3(a.T, a.heads), dim3(64), 0, st, a, q2, (float*)qn, qe);
    else hipLaunchKernelGGL(sv_latent_q_kernel<uint16_t>, dim3(a.T, a.heads), dim3(64), 0, st, a, q2, (uint16_t*)qn, qe);
}
void kr_sv_latent_direct(const KrSvLatent& a, void* qn, float* qe, bool f32, hipStream_t st) {
    if (a.T <= 0) return;
    const dim3 grid(a.T, (a.heads + 3) / 4 + (a.own_kv ? 1 : 0));
    if (f32) hipLaunchKernelGGL(sv_latent_direct_kernel<float>, grid, dim3(256), 0, st, a, (float*)qn, qe);
    else hipLaunchKernelGGL(sv_latent_direct_kernel<uint16_t>, grid, dim3(256), 0, st, a, (uint16_t*)qn, qe);
}
void kr_sv_head_rows(int T, int heads, int* seg, int* rows, int* group, hipStream_t st) {
    const int n = T * heads > heads + 1 ? T * heads : heads + 1;
    if (T <= 0) return;
    hipLaunchKernelGGL(sv_head_rows_kernel, dim3((n + 255) / 256), dim3(256), 0, st, T, heads, seg, rows, group);
}

void kr_sv_lin_scan(const KrSvLin& a, hipStream_t st) {
    if (a.T <= 0 || a.n_entries <= 0) return;
    const int dpr = (a.dim + 3) / 4;
    const dim3 grid(a.n_entries, a.heads, (a.vdim + 15) / 16);
    const size_t lds = (size_t)(((a.kind == 4 || a.kind == 7 ? 3 : 2) * 8 + 1) * 4 * dpr + 8 * 16 + 8 * 2) * sizeof(float);
#define SV_LIN(K_, DP_) hipLaunchKernelGGL((sv_lin_scan_kernel<K_, DP_>), grid, dim3(64), lds, st, a)
#define SV_LIN_D(K_) do { if (dpr <= 8) SV_LIN(K_, 8); else if (dpr <= 16) SV_LIN(K_, 16); else if (dpr <= 32) SV_LIN(K_, 32); else if (dpr <= 64) SV_LIN(K_, 64); else SV_LIN(K_, 128); } while (0)
    if (a.kind == 3) SV_LIN_D(3); else if (a.kind == 4) SV_LIN_D(4); else if (a.kind == 5) SV_LIN_D(5); else if (a.kind == 7) SV_LIN_D(7); else if (a.kind == 8) SV_LIN_D(8); else SV_LIN_D(2);
#undef SV_LIN_D
#undef SV_LIN
}
// one token per request; false: the shape is not of those (dim 32, 64 or 128 on 16-byte boundaries, at most eight waves of value columns)
bool kr_sv_lin_step(const KrSvLin& a, bool f32, hipStream_t st) {
    const int dp = a.dim / 4, ncb = (a.vdim + 15) / 16;
    if (a.kind == 5 || a.T <= 0 || a.T != a.n_entries || a.dim % 4 != 0 || (dp != 8 && dp != 16 && dp != 32) || ncb > 8 || a.rot_dims > a.dim) return false;
    if ((uintptr_t)a.state % 16 != 0 || a.state_stride % 4 != 0 || (a.kind == 3 && ((uintptr_t)a.nm % 16 != 0 || a.nm_stride % 4 != 0))) return false;
    const dim3 grid(a.T, a.heads);
#define SV_STEP(K_, DP_) hipLaunchKernelGGL((sv_lin_step_kernel<K_, DP_>), grid, dim3(64 * ncb), 0, st, a, f32)
#define SV_STEP_D(K_) do { if (dp == 8) SV_STEP(K_, 8); else if (dp == 16) SV_STEP(K_, 16); else SV_STEP(K_, 32); } while (0)
    if (a.kind == 3) SV_STEP_D(3); else if (a.kind == 4) SV_STEP_D(4); else if (a.kind == 7) SV_STEP_D(7); else if (a.kind == 8) SV_STEP_D(8); else SV_STEP_D(2);
#undef SV_STEP_D
#undef SV_STEP
    return true;
}
// the workgroup form for prompt portions of kinds 4 and 5; false: the shape does not fit its LDS buffers (the caller takes kr_sv_lin_scan)
static size_t sv_scanw_lds(int kind, int dim) {
    const int dpr = (dim + 31) / 32, dimp = 32 * ((dpr % 8 == 0) ? dpr + 4 : dpr);
    return (size_t)2 * ((kind == 4 ? 3 : 2) * 16 * dimp + 16 * 8 + 16 * 2) * sizeof(float);
}
bool kr_sv_lin_scan_wide_fits(int kind, int dim) { return (kind == 4 || kind == 5) && dim <= 512 && sv_scanw_lds(kind, dim) <= 150 * 1024; }
void kr_sv_lin_scan_wide(const KrSvLin& a, hipStream_t st) {
    if (a.T <= 0 || a.n_entries <= 0) return;
    const int dpr = (a.dim + 31) / 32;
    const dim3 grid(a.n_entries, a.heads, (a.vdim + 7) / 8);
    const size_t lds = sv_scanw_lds(a.kind, a.dim);
    if (a.kind == 4) {
        const size_t n = (size_t)a.T * a.heads * a.dim;
        hipLaunchKernelGGL(sv_gla_decay_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, const_cast<float*>(a.gz), a.gz_bias, n, a.heads * a.dim, a.inv_tau);
    }
    // one workgroup per compute unit or fewer: the pipelined walk; more: the plain one (256 compute units, up to three workgroups on each)
    const bool pipe = (size_t)grid.x * grid.y * grid.z <= 384;
#define SV_LW(K_, DP_, P_) do { if (lds > 48 * 1024 && kr_lds_optin((const void*)sv_lin_scanw_kernel<K_, DP_, P_>, lds)) return; \
                                hipLaunchKernelGGL((sv_lin_scanw_kernel<K_, DP_, P_>), grid, dim3(256), lds, st, a); } while (0)
#define SV_LW_P(K_, DP_) do { if (pipe) SV_LW(K_, DP_, true); else SV_LW(K_, DP_, false); } while (0)
#define SV_LW_D(K_) do { if (dpr <= 4) SV_LW_P(K_, 4); else if (dpr <= 8) SV_LW_P(K_, 8); else SV_LW_P(K_, 16); } while (0)
    if (a.kind == 4) SV_LW_D(4); else SV_LW_D(5);
#undef SV_LW_D
#undef SV_LW_P
#undef SV_LW
}
bool kr_sv_lin_chunked_fits(int dim, int vdim) { return dim <= 128 && vdim <= 128; }
void kr_sv_ssd_expand(const KrSvLin& a, float* z_out, int ldz, hipStream_t st) {
    if (a.T <= 0) return;
    hipLaunchKernelGGL(sv_ssd_expand_kernel, dim3(a.T, a.heads), dim3(64), 0, st, a, z_out, ldz);
}
void kr_sv_lin_chunked(const KrSvLin& a, hipStream_t st) {
    if (a.T <= 0 || a.n_entries <= 0 || a.n_chunks <= 0) return;
    const bool ml = a.kind == 3;
    const int ncb = (a.vdim + 15) / 16, ndt = (a.dim + 15) / 16, ndg = (ndt + 1) / 2;
    if (!a.prepped) hipLaunchKernelGGL(sv_lin_prep_kernel, dim3(a.T, a.heads), dim3(64), 0, st, a);
    if (ml) {
        hipLaunchKernelGGL(sv_lin_mlocal_kernel<true>, dim3(a.n_chunks, a.heads), dim3(64), 0, st, a);
        hipLaunchKernelGGL(sv_lin_mchain_kernel, dim3(a.n_entries, (a.heads + 63) / 64), dim3(64), 0, st, a);
        hipLaunchKernelGGL(sv_lin_mfinal_kernel, dim3(a.n_chunks, a.heads), dim3(64), 0, st, a);
    } else hipLaunchKernelGGL(sv_lin_mlocal_kernel<false>, dim3(a.n_chunks, a.heads), dim3(64), 0, st, a);
    const dim3 gu(a.n_chunks, a.heads, ncb * ndg);
    if (ml) hipLaunchKernelGGL((sv_lin_cupd_kernel<true, 2>), gu, dim3(64), 0, st, a);
    else hipLaunchKernelGGL((sv_lin_cupd_kernel<false, 2>), gu, dim3(64), 0, st, a);
    const dim3 gs(a.n_entries, a.heads, (a.dim * a.vdim + (ml ? a.dim : 0) + 255) / 256);
    if (ml) hipLaunchKernelGGL(sv_lin_cscan_kernel<true>, gs, dim3(256), 0, st, a);
    else hipLaunchKernelGGL(sv_lin_cscan_kernel<false>, gs, dim3(256), 0, st, a);
    kr_sv_lin_block_out(a, st);
}
void kr_sv_lin_block_out(const KrSvLin& a, hipStream_t st) {
    const bool ml = a.kind == 3;
    const dim3 go(a.n_chunks, a.heads);
    const bool small = a.dim <= 64 && a.vdim <= 64;
    const size_t lds = ((size_t)32 * (((a.vdim + 31) / 32) * 32 + 16) + (size_t)4 * (4 * ((a.dim + 15) / 16)) * 64) * sizeof(float);
    const bool whole = a.ld % 4 == 0 && (uintptr_t)a.z % 16 == 0;
    const size_t lds_whole = (size_t)32 * (a.vdim + 16) * sizeof(float);
#define SV_CO(ML_) do { if (whole && a.dim == 64 && a.vdim == 64) hipLaunchKernelGGL((sv_lin_cout_kernel<ML_, 4, 64>), go, dim3(256), lds_whole, st, a); \
                        else if (whole && a.dim == 64 && a.vdim == 128) hipLaunchKernelGGL((sv_lin_cout_kernel<ML_, 8, 64>), go, dim3(256), lds_whole, st, a); \
                        else if (whole && a.dim == 128 && a.vdim == 128) hipLaunchKernelGGL((sv_lin_cout_kernel<ML_, 8, 128>), go, dim3(256), lds_whole, st, a); \
                        else if (small) hipLaunchKernelGGL((sv_lin_cout_kernel<ML_, 4, 0>), go, dim3(256), lds, st, a); \
                        else hipLaunchKernelGGL((sv_lin_cout_kernel<ML_, 8, 0>), go, dim3(256), lds, st, a); } while (0)
    if (ml) SV_CO(true); else SV_CO(false);
#undef SV_CO
}
void kr_sv_lin_out(const KrSvLin& a, bool f32, hipStream_t st) {
    if (a.T <= 0) return;
    if (f32) hipLaunchKernelGGL(sv_lin_out_kernel<float>, dim3(a.T, a.heads), dim3(64), 0, st, a, (float*)a.out);
    else hipLaunchKernelGGL(sv_lin_out_kernel<uint16_t>, dim3(a.T, a.heads), dim3(64), 0, st, a, (uint16_t*)a.out);
}

void kr_sv_finish(const float* logits, int R, int vocab, float* const* host_logits, int* host_argmax, void* scratch, hipStream_t st) {
    if (R <= 0 || (!host_logits && !host_argmax)) return;
    const int nb = std::min(32, (vocab + 1023) / 1024), chunk = ((vocab + nb - 1) / nb + 3) / 4 * 4;
    hipLaunchKernelGGL(sv_finish_kernel, dim3(R, nb), dim3(256), 0, st, logits, vocab, chunk, host_logits, host_argmax, (unsigned long long*)scratch, (unsigned*)((unsigned long long*)scratch + R));
}

#ifdef KR_SV_STAMPS
extern "C" int kr_sv_read_stamps(long long* out16) { return hipMemcpyFromSymbol(out16, HIP_SYMBOL(sv_stamps), sizeof(long long) * 16) != hipSuccess; }
#endif
