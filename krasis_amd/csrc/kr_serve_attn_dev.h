// kr_serve_attn_dev.h -- attention of one token of a decode step on the bf16 matrix instruction, shared by its own launch (kr_serve_attn.hip, which has the reasons for the
// split operands) and by the launch that puts a product beside it (kr_serve_step.hip).
#ifndef KR_SERVE_ATTN_DEV_H
#define KR_SERVE_ATTN_DEV_H
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "kr_device.h"
#include "kr_serve_ops.h"

typedef __bf16 at_b8 __attribute__((ext_vector_type(8)));
typedef uint32_t at_u4 __attribute__((ext_vector_type(4)));
typedef uint32_t at_u2 __attribute__((ext_vector_type(2)));
constexpr float AT_LOG2E = 1.44269504f;

// two floats as three packed pairs of bf16 whose sums are the floats
__device__ __forceinline__ void at_split(float x0, float x1, uint32_t& hi, uint32_t& mid, uint32_t& lo) {
    const uint32_t a0 = __float_as_uint(x0), a1 = __float_as_uint(x1);
    hi = __builtin_amdgcn_perm(a1, a0, 0x07060302u);
    const float r0 = x0 - __uint_as_float(a0 & 0xFFFF0000u), r1 = x1 - __uint_as_float(a1 & 0xFFFF0000u);
    const uint32_t b0 = __float_as_uint(r0), b1 = __float_as_uint(r1);
    mid = __builtin_amdgcn_perm(b1, b0, 0x07060302u);
    const float s0 = r0 - __uint_as_float(b0 & 0xFFFF0000u), s1 = r1 - __uint_as_float(b1 & 0xFFFF0000u);
    lo = __builtin_amdgcn_perm(__float_as_uint(s1), __float_as_uint(s0), 0x07060302u);
}

// the waves' states [waves][rows][VDIM + 4] | [waves][16] maxima, denominators and factors | [2][16]
inline int as_lds_bytes(int heads_per_kv, int vdim, int waves) { return (waves * ((heads_per_kv < 16 ? heads_per_kv : 16) * (vdim + 4) + 3 * 16) + 32) * (int)sizeof(float); }
inline int as_lean_lds_bytes(int dim) { return 3 * 16 * (dim + 8) * 2; }      // LEAN: at least this

// Decode steps: one workgroup (eight waves in a launch of its own) per (token, key / value head, 16 query heads of its group, share of the keys).  A wave takes 32 keys at a time on
// v_mfma_f32_16x16x32_bf16 with the operands split as above, keys and values straight from the cache to registers (a row serves one token's heads only: nothing to share):
//   S^T[key][row] = K Q^T    first operand: 16 key rows, a lane 16 bytes of a row;
//   O^T[d][row] += V^T P^T   a lane holds the 8 keys (4 q + 0..3 of both blocks of 16) that its weights belong to, VDIM / 16 neighbouring columns each; byte permutes turn
//                            them into the columns' fragments, column 16-row d of block j = d VDIM / 16 + j.
// What it waits for is latency -- page table, rows, two short products, one merge through LDS -- so a wave requests keys and values together, the next 32 keys before it works on
// these.  32 keys lie in one page (the page size is a multiple of 32).  One request, 16 / 2 heads of 128: 20.9 us on the f32 matrix instruction -> 7.3 at some 110 keys.
// bx: token, by: key / value head, bz: share of the keys and batch of 16 query heads; lds: as_lds_bytes; NW: waves.
// LEAN: half the registers (128 at head size 128, which leaves four waves to a SIMD for what runs beside it): the query's pieces stay in LDS and the next keys are
// requested when these are done with, which a wave with one batch of keys never notices.
template <int DIM, int VDIM, int NW, bool LEAN = false>
__device__ __forceinline__ void as_token(const KrSvAttn& a, const int bx, const int by, const int bz, float* lds) {
    constexpr int KS = DIM / 32, CPL = VDIM / 16, VW = CPL / 2;
    const int R = a.heads / a.kv_heads, t = a.toks ? a.toks[bx] : bx, g = by, hb = __builtin_amdgcn_readfirstlane(bz / a.nsplit), sp = bz - hb * a.nsplit;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), row = lane & 15, q = lane >> 4;
    const int Rb = min(16, R - hb * 16), h0 = g * R + hb * 16, head = h0 + min(row, Rb - 1);
    const int p = a.pos[t];
    const int* table = a.page_table + (size_t)a.slot[t] * a.table_ld;
    const int lo = a.window > 0 ? max(0, p - a.window + 1) : (a.chunk > 0 ? p - p % a.chunk : 0);
    // kept first keys: their own leading tiles when the window's tiles, which begin at a multiple of 32, lie past the last of them (else that tile would hold kept keys too, and
    // the mask lets them through wherever they stand), else one contiguous range from 0
    const int nck = a.keep > 0 && (lo & ~31) >= a.keep ? (a.keep + 31) / 32 : 0;
    const int first = a.keep > 0 && nck == 0 ? 0 : lo & ~31;
    const int nch = (p - first) / 32 + 1 + nck, cps = __builtin_amdgcn_readfirstlane((nch + a.nsplit - 1) / a.nsplit), c0 = sp * cps, c1 = min(nch, c0 + cps);
    at_u4 kn[2][KS]; uint32_t vn[8][VW];
    auto request = [&](int c) {
        const int j0 = c < nck ? 32 * c : first + 32 * (c - nck), jl = (c < nck ? a.keep - 1 : p) - j0;      // keys past the last one are fetched again and masked
        // 32 keys lie in one page: the base is the wave's, a lane adds a 32-bit offset (quotients come from the vector unit, hence readfirstlane)
        const int page = __builtin_amdgcn_readfirstlane(j0 / a.page_tokens);
        const size_t base = (size_t)table[page] * a.page_tokens + (j0 - page * a.page_tokens);
        const uint16_t* kp = (const uint16_t*)a.kpool + base * a.ldk + (size_t)g * DIM;
        const uint16_t* vp = (const uint16_t*)a.vpool + base * a.ldv + (size_t)g * VDIM;
#pragma unroll
        for (int b = 0; b < 2; b++) {
            const uint32_t k = min(b * 16 + row, jl) * a.ldk + q * 8;
#pragma unroll
            for (int ks = 0; ks < KS; ks++) kn[b][ks] = *reinterpret_cast<const at_u4*>(kp + (k + ks * 32));
        }
#pragma unroll
        for (int i = 0; i < 8; i++) {
            const uint16_t* v = vp + (uint32_t)(min((i >> 2) * 16 + 4 * q + (i & 3), jl) * a.ldv + row * CPL);
            if constexpr (VW == 1) vn[i][0] = *reinterpret_cast<const uint32_t*>(v);
            else if constexpr (VW == 2) { const at_u2 x = *reinterpret_cast<const at_u2*>(v); vn[i][0] = x.x; vn[i][1] = x.y; }
            else {
#pragma unroll
                for (int u = 0; u < VW / 4; u++) {
                    const at_u4 x = *reinterpret_cast<const at_u4*>(v + 8 * u);
#pragma unroll
                    for (int e = 0; e < 4; e++) vn[i][4 * u + e] = x[e];
                }
            }
        }
    };
    if (c0 + wave < c1) request(c0 + wave);
    at_u4 qh[KS], qm[KS], ql[KS];
    constexpr int QS = DIM + 8;
    uint16_t* lq = (uint16_t*)lds;           // LEAN: [3][16][QS] pieces of the query rows, where the waves' states meet later
    if constexpr (LEAN) {
        const float qscale = a.softcap > 0.0f ? a.scale : a.scale * AT_LOG2E;
        for (int i = tid; i < 16 * DIM / 8; i += 64 * NW) {
            const int r = i / (DIM / 8), k = (i - r * (DIM / 8)) * 8;
            const float* qp = a.qkv + (size_t)t * a.ldq + (size_t)(h0 + min(r, Rb - 1)) * DIM + k;
            float v[8];
            *reinterpret_cast<float4*>(&v[0]) = *reinterpret_cast<const float4*>(qp);
            *reinterpret_cast<float4*>(&v[4]) = *reinterpret_cast<const float4*>(qp + 4);
            at_u4 x, y, z;
#pragma unroll
            for (int e = 0; e < 4; e++) {
                uint32_t hi, mid, lo;
                at_split(v[2 * e] * qscale, v[2 * e + 1] * qscale, hi, mid, lo);
                x[e] = hi; y[e] = mid; z[e] = lo;
            }
            *reinterpret_cast<at_u4*>(&lq[r * QS + k]) = x; *reinterpret_cast<at_u4*>(&lq[(16 + r) * QS + k]) = y; *reinterpret_cast<at_u4*>(&lq[(32 + r) * QS + k]) = z;
        }
        __syncthreads();
    } else {
        const float qscale = a.softcap > 0.0f ? a.scale : a.scale * AT_LOG2E;
        const float* qp = a.qkv + (size_t)t * a.ldq + (size_t)head * DIM + q * 8;
#pragma unroll
        for (int ks = 0; ks < KS; ks++) {
            float v[8];
            *reinterpret_cast<float4*>(&v[0]) = *reinterpret_cast<const float4*>(qp + ks * 32);
            *reinterpret_cast<float4*>(&v[4]) = *reinterpret_cast<const float4*>(qp + ks * 32 + 4);
#pragma unroll
            for (int i = 0; i < 4; i++) {
                uint32_t x, y, z;
                at_split(v[2 * i] * qscale, v[2 * i + 1] * qscale, x, y, z);
                qh[ks][i] = x; qm[ks][i] = y; ql[ks][i] = z;
            }
        }
    }
    const float slope = a.slopes ? a.slopes[head] * AT_LOG2E : 0.0f;
    typedef float at_f4 __attribute__((ext_vector_type(4)));
    float m = -INFINITY, l = 0.0f;
    at_f4 acc[CPL];
#pragma unroll
    for (int j = 0; j < CPL; j++) acc[j] = at_f4{0.0f, 0.0f, 0.0f, 0.0f};
    for (int c = c0 + wave; c < c1; c += NW) {
        at_u4 kv[2][KS]; uint32_t vv[8][VW];
#pragma unroll
        for (int b = 0; b < 2; b++)
#pragma unroll
            for (int ks = 0; ks < KS; ks++) kv[b][ks] = kn[b][ks];
#pragma unroll
        for (int i = 0; i < 8; i++)
#pragma unroll
            for (int u = 0; u < VW; u++) vv[i][u] = vn[i][u];
        if (!LEAN && c + NW < c1) request(c + NW);
        const int j0 = c < nck ? 32 * c : first + 32 * (c - nck), jl = c < nck ? a.keep - 1 : p;
        at_f4 st[2];
#pragma unroll
        for (int b = 0; b < 2; b++) st[b] = at_f4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int ks = 0; ks < KS; ks++) {
            if constexpr (LEAN) {
                int at0 = row * QS + q * 8 + ks * 32;
                asm volatile("" : "+v"(at0));            // else the reads leave the loop, for as many registers as they were to save
                const uint16_t* at = lq + at0;
                qh[ks] = *reinterpret_cast<const at_u4*>(at); qm[ks] = *reinterpret_cast<const at_u4*>(at + 16 * QS); ql[ks] = *reinterpret_cast<const at_u4*>(at + 32 * QS);
            }
#pragma unroll
            for (int b = 0; b < 2; b++) st[b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(at_b8, kv[b][ks]), __builtin_bit_cast(at_b8, ql[ks]), st[b], 0, 0, 0);
#pragma unroll
            for (int b = 0; b < 2; b++) st[b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(at_b8, kv[b][ks]), __builtin_bit_cast(at_b8, qm[ks]), st[b], 0, 0, 0);
#pragma unroll
            for (int b = 0; b < 2; b++) st[b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(at_b8, kv[b][ks]), __builtin_bit_cast(at_b8, qh[ks]), st[b], 0, 0, 0);
        }
        float cm = -INFINITY;
#pragma unroll
        for (int b = 0; b < 2; b++)
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const int key = j0 + b * 16 + 4 * q + i;
                float sc = st[b][i];
                if (a.softcap > 0.0f) sc = a.softcap * tanhf(sc / a.softcap) * AT_LOG2E;
                if (a.slopes) sc -= slope * (float)(p - key);
                const bool ok = (key <= jl) & ((key >= lo) | (key < a.keep));
                st[b][i] = ok ? sc : -INFINITY;
                cm = fmaxf(cm, st[b][i]);
            }
        cm = fmaxf(cm, __shfl_xor(cm, 16)); cm = fmaxf(cm, __shfl_xor(cm, 32));
        const float mn = fmaxf(m, cm), base = mn == -INFINITY ? 0.0f : mn, alpha = __builtin_amdgcn_exp2f(m - base);
        m = mn; l *= alpha;
#pragma unroll
        for (int b = 0; b < 2; b++)
#pragma unroll
            for (int i = 0; i < 4; i++) { const float e = __builtin_amdgcn_exp2f(st[b][i] - base); st[b][i] = e; l += e; }
        at_u4 ph, pm, pl;
#pragma unroll
        for (int i = 0; i < 4; i++) {
            uint32_t x, y, z;
            at_split(st[i >> 1][2 * (i & 1)], st[i >> 1][2 * (i & 1) + 1], x, y, z);
            ph[i] = x; pm[i] = y; pl[i] = z;
        }
#pragma unroll
        for (int j = 0; j < CPL; j++) {
            at_u4 vf;
#pragma unroll
            for (int e = 0; e < 4; e++) vf[e] = __builtin_amdgcn_perm(vv[2 * e + 1][j >> 1], vv[2 * e][j >> 1], (j & 1) ? 0x07060302u : 0x05040100u);
            acc[j] *= alpha;
            acc[j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(at_b8, vf), __builtin_bit_cast(at_b8, pl), acc[j], 0, 0, 0);
            acc[j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(at_b8, vf), __builtin_bit_cast(at_b8, pm), acc[j], 0, 0, 0);
            acc[j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(at_b8, vf), __builtin_bit_cast(at_b8, ph), acc[j], 0, 0, 0);
        }
        if (LEAN && c + NW < c1) request(c + NW);
    }
    // ---- the waves' states meet: [waves][Rb][VDIM + 4] sums | [waves][16] maxima | [waves][16] denominators | [waves][16] factors | [16] 1 / denominator, [16] maximum
    constexpr int VS = VDIM + 4;
    float* ml = lds + NW * Rb * VS; float* dl = ml + NW * 16; float* fl = dl + NW * 16; float* rl = fl + NW * 16;
    l += __shfl_xor(l, 16); l += __shfl_xor(l, 32);
    if (LEAN) __syncthreads();               // every wave is past its last read of the query
    if (q == 0) { ml[wave * 16 + row] = m; dl[wave * 16 + row] = l; }
    if (row < Rb) {
#pragma unroll
        for (int j = 0; j < CPL; j++)
#pragma unroll
            for (int i = 0; i < 4; i++) lds[(wave * Rb + row) * VS + (4 * q + i) * CPL + j] = acc[j][i];
    }
    __syncthreads();
    const bool last = a.nsplit == 1;
    if (tid < NW * 16) {
        const int w = tid >> 4, r = tid & 15;
        const float sk = last && a.sink && r < Rb ? a.sink[h0 + r] * AT_LOG2E : -INFINITY;
        float M = sk;
#pragma unroll
        for (int i = 0; i < NW; i++) M = fmaxf(M, ml[i * 16 + r]);
        fl[tid] = ml[tid] == -INFINITY ? 0.0f : exp2f(ml[tid] - M);
        if (w == 0) {
            float L = last && a.sink && r < Rb ? exp2f(sk - M) : 0.0f;
            for (int i = 0; i < NW; i++) { const float mw = ml[i * 16 + r]; if (mw != -INFINITY) L += dl[i * 16 + r] * exp2f(mw - M); }
            rl[r] = last ? 1.0f / L : L; rl[16 + r] = M;
        }
    }
    __syncthreads();
    for (int i = tid; i < Rb * VDIM; i += 64 * NW) {
        const int r = i / VDIM, c = i - r * VDIM, h = h0 + r;
        float v = 0.0f;
#pragma unroll
        for (int w = 0; w < NW; w++) v = __builtin_fmaf(lds[(w * Rb + r) * VS + c], fl[w * 16 + r], v);
        if (last) {
            const float gt = a.out_gate ? 1.0f / (1.0f + expf(-a.out_gate[(size_t)t * a.ld_gate + (a.gate_elem ? (size_t)h * VDIM + c : (size_t)h)])) : 1.0f;
            ((uint16_t*)a.out)[(size_t)t * (a.out_ld ? a.out_ld : a.heads * VDIM) + (size_t)h * VDIM + c] = kr_f32_to_bf16(v * rl[r] * gt * (a.out_scale != 0.0f ? a.out_scale : 1.0f));
        } else {
            const size_t slot = ((size_t)bx * a.heads + h) * a.nsplit + sp;
            a.part_acc[slot * VDIM + c] = v;
            if (c == 0) { a.part_ml[slot * 2] = rl[16 + r]; a.part_ml[slot * 2 + 1] = rl[r]; }
        }
    }
}

#endif
