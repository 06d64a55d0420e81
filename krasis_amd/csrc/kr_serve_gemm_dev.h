// kr_serve_gemm_dev.h -- what the matrix products of the batched serving step share on the device: element conversion, the epilogue of one element of C,
// the gated activation, and the row tile of a grouped problem.
#ifndef KR_SERVE_GEMM_DEV_H
#define KR_SERVE_GEMM_DEV_H
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "kr_device.h"
#include "kr_serve_ops.h"

typedef float gv16f __attribute__((ext_vector_type(16)));
typedef __bf16 gb8 __attribute__((ext_vector_type(8)));
typedef uint32_t gu4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ float gm_ld(const float* p) { return *p; }
__device__ __forceinline__ float gm_ld(const uint16_t* p) { return kr_bf16_to_f32(*p); }
// one element of C: f32, or the storage type when the output feeds another GEMM as it is (BF = a bf16 store)
template <bool BF>
__device__ __forceinline__ void gm_store(const KrSvGemm& g, int m, int n, float v, float* host = nullptr) {
    const int row = g.c_rows ? g.c_rows[m] : m;
    const size_t i = (size_t)row * g.ldc + n;
    if (g.bias) v += g.bias[n];
    if (n >= g.silu_lo && n < g.silu_hi) v = v / (1.0f + expf(-v));
    if (g.o_gate) v *= 1.0f / (1.0f + expf(-g.o_gate[(size_t)(row / g.o_gate_div) * g.o_gate_ld + (size_t)(row % g.o_gate_div) * g.N + n]));
    if (BF && g.c_storage) ((uint16_t*)g.C)[i] = kr_f32_to_bf16(v);
    else {
        g.C[i] = v;
        if (BF && host) host[i] = v;
    }
}

// where a step's arrays say that its results go (KrSvGemm::c_host, sv_finish); a scalar load: the word does not change while a launch runs
__device__ __forceinline__ float* gm_host(float* const* at) { return at ? (float*)*(const __attribute__((address_space(4))) uint64_t*)(uintptr_t)at : nullptr; }
// columns of group `group`: all N, or what the group's own matrix has
__device__ __forceinline__ int gm_cols(const KrSvGemm& g, int group) { return g.n_last > 0 ? (group == g.n_groups - 1 ? g.n_last : g.n_first) : g.N; }

// row tile `tile` of a grouped problem: false past the last tile.  The groups' tile counts go through a prefix sum over the lanes, 64 groups at a time (a walk
// from group to group is a chain of dependent loads, up to 128 of them before a tile of the last expert could begin).  All lanes of a wave call it.
__device__ __forceinline__ bool gm_find_tile(const int* seg, int n_groups, int tile, int BM, int& group, int& m0, int& mend) {
    const int lane = threadIdx.x & 63;
    int acc = 0;
    for (int g0 = 0; g0 < n_groups; g0 += 64) {
        const int g = min(g0 + lane, n_groups - 1);
        const int lo = seg[g], hi = seg[g + 1];
        const int nt = g0 + lane < n_groups ? (hi - lo + BM - 1) / BM : 0;
        int sum = nt;                                    // tiles of the groups up to and with this lane's
#pragma unroll
        for (int o = 1; o < 64; o <<= 1) { const int v = __shfl_up(sum, o); if (lane >= o) sum += v; }
        const unsigned long long mine = __ballot(tile < acc + sum);
        if (mine) {
            const int l = __ffsll(mine) - 1;
            group = __builtin_amdgcn_readfirstlane(g0 + l);
            m0 = __builtin_amdgcn_readfirstlane(__shfl(lo, l) + (tile - acc - __shfl(sum - nt, l)) * BM);
            mend = __builtin_amdgcn_readfirstlane(__shfl(hi, l));
            return true;
        }
        acc += __shfl(sum, 63);
    }
    return false;
}

__device__ __forceinline__ float gm_act(float g, float u, int kind, float limit, float alpha) {
    if (kind == KR_SV_ACT_RELU2) { g = fmaxf(g, 0.0f); return g * g; }
    if (kind == KR_SV_ACT_GELU_TANH) return 0.5f * g * (1.0f + tanhf(0.7978845608028654f * (g + 0.044715f * g * g * g))) * u;
    if (kind == KR_SV_ACT_CLAMPED_SWIGLU) { g = fminf(g, limit); u = fminf(fmaxf(u, -limit), limit); return g / (1.0f + expf(-alpha * g)) * (u + 1.0f); }
    // silu on the hardware exponential and reciprocal (one ulp each): every wave of a decode step's down projection forms it again
    return g * __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(-1.4426950408889634f * g)) * u;
}
// the same where every element is formed once
__device__ __forceinline__ float gm_act_once(float g, float u, int kind, float limit, float alpha) {
    if (kind == KR_SV_ACT_RELU2 || kind == KR_SV_ACT_GELU_TANH || kind == KR_SV_ACT_CLAMPED_SWIGLU) return gm_act(g, u, kind, limit, alpha);
    return g / (1.0f + expf(-g)) * u;
}
template <typename T> __device__ __forceinline__ float gm_round(float v) { return v; }
template <> __device__ __forceinline__ float gm_round<uint16_t>(float v) { return kr_bf16_to_f32(kr_f32_to_bf16(v)); }

#endif
