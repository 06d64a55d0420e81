// kr_serve_attn.hip -- attention of a bf16 store on the bf16 matrix instruction, every operand exact: prompt portions, and decode steps further down.
//
// Scores and weights of this design are 32-bit numbers, the cache holds bf16.  A 32-bit float is the exact sum of three bf16 numbers (24 bits of significand = 8 + 8 + 8,
// taken by truncation), so q K^T = (q_hi + q_mid + q_lo) K^T and P V alike are three passes of the bf16 instruction with f32 accumulators: no operand loses a bit, and
// three passes at sixteen times the rate of v_mfma_f32_16x16x4_f32 take a fifth of its time.
//
// A workgroup owns 128 query ROWS of one request that share a key / value head: the heads of the group for 128 / R consecutive tokens; wave w rows 32 w .. 32 w + 31.
// Keys come in tiles of 64, K and V by LDS-DMA into two slots each (the next tile is requested before the current one is used, one barrier per tile).  Both products are
// formed transposed,
//   S^T[key][row] = K Q^T     (first operand: key rows from LDS; second: the row's query pieces, in registers for the whole launch)
//   O^T[d][row]  += V^T P^T   (first operand: value columns by the transposing LDS read; second: the weights exactly where the first product left them)
// so a lane's accumulators belong to ONE row (lane % 32), the softmax is per lane, and the two halves of a wave only exchange the row's maximum.  The reduction index of
// the second product is permuted to the order in which a lane holds its keys (4 h + 0..3, 8 + 4 h + 0..3 of a block of 16 for wave half h).
// LDS-DMA writes lane-linear, so the chunk order is swizzled on the source side: K chunk c of row r at c ^ (r / rows per 256 bytes), V groups of four chunks likewise, which
// spreads the 32 rows of a fragment read, and the 4 rows x 64 bytes of a transposing read, over all banks.
// Bound: the matrix instruction, three times 4 H D keys operations (about 50 us at the case below); exponentials, the splitting of the weights and the addresses (some 700
// vector instructions per tile and wave beside 96 products) run beside it in the SIMD's other wave.  Per launch, us, f32 matrix instruction before -> now: 4096 tokens, 16 / 2 heads
// of 128, window 1024: 490 -> 108; 3300 tokens of three requests, 64 / 4 heads, window 2048: 1230 -> 249.  64-bit oracle of a whole prompt: error 5.1e-3 before, 4.4e-3
// now (the store's bf16 roundings).
#include <hip/hip_runtime.h>
#include <stdint.h>
#include <algorithm>

#include "kr_device.h"
#include "kr_lds_optin.h"
#include "kr_serve_attn_dev.h"
#include "kr_serve_ops.h"

namespace {
typedef float at_f16 __attribute__((ext_vector_type(16)));
constexpr int AT_KEYS = 64, AT_ROWS = 128;

__device__ __forceinline__ uint32_t at_lds_addr(const void* p) { return (uint32_t)(uintptr_t)(const __attribute__((address_space(3))) char*)p; }
// 64 lanes x 16 bytes from the lane's own address to lds_dst (wave-uniform) + 16 lane; M0 is the compiler's register.  Not counted by the compiler: see the wait below.
__device__ __forceinline__ void at_dma16(uint32_t lds_dst, const uint16_t* src) {
    unsigned keep;
    asm volatile("s_mov_b32 %0, m0\n\ts_mov_b32 m0, %2\n\ts_nop 2\n\tglobal_load_lds_dwordx4 %1, off\n\ts_mov_b32 m0, %0" : "=&s"(keep) : "v"(src), "s"(lds_dst) : "memory");
}
__device__ __forceinline__ void at_wait_barrier() { asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

__device__ __forceinline__ float at_other_half(float x, int h) {
    const uint32_t u = __float_as_uint(x);
    const auto sw = __builtin_amdgcn_permlane32_swap(u, u, false, false);
    return __uint_as_float(h ? sw[0] : sw[1]);
}

template <int DIM, int VDIM>
__global__ void __launch_bounds__(256, 2) sv_attn_prompt_kernel(const KrSvAttn a) {
    constexpr int KC = DIM / 8, VC = VDIM / 8;                 // 16-byte chunks of a cache row's head
    constexpr int KS = DIM / 16, DB = VDIM / 32;               // k steps of the first product, column blocks of the second
    constexpr int KRQ = 64 / KC, VRQ = 64 / VC;                // rows per request
    constexpr int KREQ = 16 / KRQ, VREQ = 16 / VRQ;            // requests of a wave per tile: it brings rows 16 w .. 16 w + 15
    constexpr int KSLOT = AT_KEYS * DIM, VSLOT = AT_KEYS * VDIM;
    constexpr int KRP = 16 / KC, VRP = 16 / VC;                // rows per 256 bytes
    __shared__ __attribute__((aligned(1024))) uint16_t Kt[2 * KSLOT];
    __shared__ __attribute__((aligned(1024))) uint16_t Vt[2 * VSLOT];
    // The last pieces of the first LQ k steps wait in LDS, each lane's its own.  At 128 x 128 the query pieces, sums and scores of two waves per SIMD were 25 registers more than
    // there are, and a reload of a spilled one waits, in order, for the next tile's rows requested before it: 4096 tokens 140 us a launch with the spills, 108 without, 3300 of
    // three requests 326 / 249.
    constexpr int LQ = DIM == 128 && VDIM == 128 ? 4 : 0;
    __shared__ at_u4 Lq[LQ > 0 ? 4 * LQ * 64 : 1];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), n = lane & 31, h = lane >> 5;
    const int R = a.heads / a.kv_heads, TQ = AT_ROWS / R, g = blockIdx.y, sp = blockIdx.z;
    // the tile of tokens: entries' tile counts (short entries may have a launch of their own) through a prefix sum over the lanes
    int t0 = 0, cnt = 0;
    {
        int acc = 0;
        bool found = false;
        for (int e0 = 0; e0 < a.n_entries && !found; e0 += 64) {
            const int e = min(e0 + lane, a.n_entries - 1);
            const int lo = a.ent_off[e], hi = a.ent_off[e + 1], nt = e0 + lane < a.n_entries && hi - lo > a.few ? (hi - lo + TQ - 1) / TQ : 0;
            int sum = nt;
#pragma unroll
            for (int o = 1; o < 64; o <<= 1) { const int v = __shfl_up(sum, o); if (lane >= o) sum += v; }
            const unsigned long long mine = __ballot((int)blockIdx.x < acc + sum);
            if (mine) {
                const int l = __ffsll(mine) - 1, first = __shfl(lo, l) + ((int)blockIdx.x - acc - __shfl(sum - nt, l)) * TQ;
                t0 = __builtin_amdgcn_readfirstlane(first);
                cnt = __builtin_amdgcn_readfirstlane(min(TQ, __shfl(hi, l) - first));
                found = true;
            }
            acc += __shfl(sum, 63);
        }
        if (!found) return;
    }
    const int row = wave * 32 + n, tq = row / R, head = g * R + row % R;
    const bool rv = tq < cnt;
    const int p0 = a.pos[t0], sl = a.slot[t0];
    const int p_row = rv ? p0 + tq : -1;
    const int lo_row = a.window > 0 ? max(0, p_row - a.window + 1) : (a.chunk > 0 && rv ? p_row - p_row % a.chunk : 0);
    const int keep_row = rv ? a.keep : 0;
    const float slope = (a.slopes && rv) ? a.slopes[head] * AT_LOG2E : 0.0f;
    const int hi = p0 + cnt - 1;
    int lo = a.window > 0 ? max(0, p0 - a.window + 1) : (a.chunk > 0 ? p0 - p0 % a.chunk : 0);
    // kept first keys: their own leading tiles when every row's window has left them behind, else one contiguous range from 0
    const int nck = a.keep > 0 && lo > a.keep ? (a.keep + AT_KEYS - 1) / AT_KEYS : 0;
    if (a.keep > 0 && nck == 0) lo = 0;
    const int nch = (hi - lo) / AT_KEYS + 1 + nck, cps = (nch + a.nsplit - 1) / a.nsplit, c0 = sp * cps, c1 = min(nch, c0 + cps);
    // what this wave's rows can see (wave-uniform): tiles outside are only brought in, tiles inside need no mask
    const int wt0 = wave * 32 / R, wt1 = min(cnt - 1, (wave * 32 + 31) / R);
    const bool w_any = wt0 < cnt;
    const int wp0 = p0 + wt0, wp1 = p0 + wt1;                  // first and last position among the rows
    const int wlo = a.window > 0 ? max(0, wp0 - a.window + 1) : (a.chunk > 0 ? wp0 - wp0 % a.chunk : 0);      // first key any row sees beside the kept ones
    const int wlo1 = a.window > 0 ? max(0, wp1 - a.window + 1) : (a.chunk > 0 ? wp1 - wp1 % a.chunk : 0);     // first key every row sees
    const bool w_full = (wave * 32 + 31) / R < cnt;
    // ---- the rows' queries, scaled, in three pieces: k step ks holds dims of chunk ks + KS h.  Scores are kept in powers of two (one factor, one rounding as before): an
    // exponential is then one subtraction and one hardware instruction
    const float qscale = a.softcap > 0.0f ? a.scale : a.scale * AT_LOG2E;
    at_u4 qh[KS], qm[KS], ql[KS];
    const int lq0 = wave * LQ * 64 + lane;
    {
        const float* qp = a.qkv + (size_t)(t0 + (rv ? tq : 0)) * a.ldq + (size_t)head * DIM + (size_t)(KS * h) * 8;
#pragma unroll
        for (int ks = 0; ks < KS; ks++) {
            float v[8];
            *reinterpret_cast<float4*>(&v[0]) = *reinterpret_cast<const float4*>(qp + ks * 8);
            *reinterpret_cast<float4*>(&v[4]) = *reinterpret_cast<const float4*>(qp + ks * 8 + 4);
#pragma unroll
            for (int i = 0; i < 4; i++) {
                uint32_t x, y, z;
                at_split(rv ? v[2 * i] * qscale : 0.0f, rv ? v[2 * i + 1] * qscale : 0.0f, x, y, z);
                qh[ks][i] = x; qm[ks][i] = y; ql[ks][i] = z;
            }
            if (ks < LQ) Lq[lq0 + ks * 64] = ql[ks];
        }
    }
    const int* table = a.page_table + (size_t)sl * a.table_ld;
    const uint16_t* kp = (const uint16_t*)a.kpool + (size_t)g * DIM;
    const uint16_t* vp = (const uint16_t*)a.vpool + (size_t)g * VDIM;
    const uint32_t kdst = __builtin_amdgcn_readfirstlane(at_lds_addr(Kt)) + (uint32_t)wave * (16 * DIM * 2), vdst = __builtin_amdgcn_readfirstlane(at_lds_addr(Vt)) + (uint32_t)wave * (16 * VDIM * 2);
    auto tile_at = [&](int c, int& j0, int& jl) { j0 = c < nck ? AT_KEYS * c : lo + AT_KEYS * (c - nck); jl = c < nck ? a.keep - 1 : hi; };
    // the pool row of key j0 + lane of tile c (keys past the last one: the last one, masked later): read a tile ahead of the requests that need it
    auto rows_of = [&](int c) {
        int j0, jl;
        tile_at(c, j0, jl);
        const int key = min(j0 + lane, jl), page = key / a.page_tokens;
        return table[page] * a.page_tokens + (key - page * a.page_tokens);
    };
    auto request = [&](int prow, int slot) {
#pragma unroll
        for (int i = 0; i < KREQ; i++) {
            const int pr = __shfl(prow, wave * 16 + i * KRQ + lane / KC);
            const int r = wave * 16 + i * KRQ + lane / KC, ch = (lane % KC) ^ ((r / KRP) % KC);
            at_dma16(kdst + (uint32_t)(slot * KSLOT * 2 + i * 1024), kp + (size_t)pr * a.ldk + ch * 8);
        }
#pragma unroll
        for (int i = 0; i < VREQ; i++) {
            const int pr = __shfl(prow, wave * 16 + i * VRQ + lane / VC);
            const int r = wave * 16 + i * VRQ + lane / VC, ch = (lane % VC) ^ (4 * ((r / VRP) % (VC / 4)));
            at_dma16(vdst + (uint32_t)(slot * VSLOT * 2 + i * 1024), vp + (size_t)pr * a.ldv + ch * 8);
        }
    };
    float m = -INFINITY, l = 0.0f;                             // l: this lane's keys only; the halves meet at the end
    at_f16 acc[DB];
#pragma unroll
    for (int d = 0; d < DB; d++)
#pragma unroll
        for (int i = 0; i < 16; i++) acc[d][i] = 0.0f;
    if (c0 < c1) request(rows_of(c0), 0);
    int next = c0 + 1 < c1 ? rows_of(c0 + 1) : 0;
    for (int c = c0; c < c1; c++) {
        const int slot = (c - c0) & 1;
        at_wait_barrier();                                     // the tile has landed for every wave, and the other slot's reads are over
        if (c + 1 < c1) request(next, slot ^ 1);
        if (c + 2 < c1) next = rows_of(c + 2);
        int j0, jl;
        tile_at(c, j0, jl);
        const int je = min(j0 + AT_KEYS - 1, jl);              // last real key of the tile
        if (!w_any || j0 > wp1 || (je < wlo && j0 >= a.keep)) continue;
        int nk = n, lv = lane;                                 // (addresses of fragments are formed per tile: hoisted, they are what spills)
        if (LQ > 0) asm volatile("" : "+v"(nk), "+v"(lv));
        // ---- S^T: two blocks of 32 keys
        at_f16 st[2];
#pragma unroll
        for (int b = 0; b < 2; b++)
#pragma unroll
            for (int i = 0; i < 16; i++) st[b][i] = 0.0f;
#pragma unroll
        for (int ks = 0; ks < KS; ks++) {
            at_b8 kf[2];
            if (ks < LQ) {
                int at = lq0 + ks * 64;
                asm volatile("" : "+v"(at));                   // else the read leaves the loop, for the register it was to save
                ql[ks] = Lq[at];
            }
#pragma unroll
            for (int b = 0; b < 2; b++) kf[b] = __builtin_bit_cast(at_b8, *reinterpret_cast<const at_u4*>(&Kt[slot * KSLOT + (b * 32 + nk) * DIM + (((ks + KS * h) ^ (((b * 32 + nk) / KRP) % KC)) * 8)]));
#pragma unroll
            for (int b = 0; b < 2; b++) st[b] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kf[b], __builtin_bit_cast(at_b8, ql[ks]), st[b], 0, 0, 0);
#pragma unroll
            for (int b = 0; b < 2; b++) st[b] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kf[b], __builtin_bit_cast(at_b8, qm[ks]), st[b], 0, 0, 0);
#pragma unroll
            for (int b = 0; b < 2; b++) st[b] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kf[b], __builtin_bit_cast(at_b8, qh[ks]), st[b], 0, 0, 0);
        }
        // ---- capped scores, distance bias, masks
        if (a.softcap > 0.0f) {
#pragma unroll
            for (int b = 0; b < 2; b++)
#pragma unroll
                for (int i = 0; i < 16; i++) st[b][i] = a.softcap * tanhf(st[b][i] / a.softcap) * AT_LOG2E;
        }
        const int key0 = j0 + 4 * h;                           // key of st[b][i]: key0 + 32 b + (i & 3) + 8 (i >> 2)
        if (a.slopes) {
#pragma unroll
            for (int b = 0; b < 2; b++)
#pragma unroll
                for (int i = 0; i < 16; i++) st[b][i] -= slope * (float)(p_row - (key0 + 32 * b + (i & 3) + 8 * (i >> 2)));
        }
        if (!(w_full && j0 + AT_KEYS - 1 <= min(wp0, jl) && j0 >= wlo1)) {
            const int last = rv ? min(p_row, jl) : -1;
#pragma unroll
            for (int b = 0; b < 2; b++)
#pragma unroll
                for (int i = 0; i < 16; i++) {
                    const int key = key0 + 32 * b + (i & 3) + 8 * (i >> 2);
                    const bool ok = (key <= last) & ((key >= lo_row) | (key < keep_row));
                    st[b][i] = ok ? st[b][i] : -INFINITY;
                }
        }
        // ---- online softmax of this lane's row
        float cm = -INFINITY;
#pragma unroll
        for (int b = 0; b < 2; b++)
#pragma unroll
            for (int i = 0; i < 16; i++) cm = fmaxf(cm, st[b][i]);
        cm = fmaxf(cm, at_other_half(cm, h));
        const float mn = fmaxf(m, cm);
        const float base = mn == -INFINITY ? 0.0f : mn;        // a row that has seen no key yet keeps its zero state
        const float alpha = __builtin_amdgcn_exp2f(m - base);
        m = mn;
        if (__any(alpha != 1.0f)) {
            l *= alpha;
#pragma unroll
            for (int d = 0; d < DB; d++) acc[d] *= alpha;
        }
#pragma unroll
        for (int b = 0; b < 2; b++)
#pragma unroll
            for (int i = 0; i < 16; i++) { const float p = __builtin_amdgcn_exp2f(st[b][i] - base); st[b][i] = p; l += p; }
        // ---- O^T += V^T P^T: blocks of 16 keys
#pragma unroll
        for (int kt = 0; kt < 4; kt++) {
            at_u4 ph, pm, pl;
#pragma unroll
            for (int i = 0; i < 4; i++) {
                uint32_t x, y, z;
                at_split(st[kt >> 1][8 * (kt & 1) + 2 * i], st[kt >> 1][8 * (kt & 1) + 2 * i + 1], x, y, z);
                ph[i] = x; pm[i] = y; pl[i] = z;
            }
            typedef __fp16 at_h4 __attribute__((__vector_size__(4 * sizeof(__fp16))));
            const int r = 16 * kt + 4 * h + ((lv & 15) >> 2);          // this lane points at row r (and r + 8), four columns of its 16-lane group
            at_b8 vf[DB];
#pragma unroll
            for (int d = 0; d < DB; d++) {
                const int col = 32 * d + 16 * ((lv >> 4) & 1) + 4 * (lv & 3);
                const uint16_t* v0 = &Vt[slot * VSLOT + r * VDIM + (((col >> 3) ^ (4 * ((r / VRP) % (VC / 4)))) * 8) + (col & 7)];
                const uint16_t* v1 = &Vt[slot * VSLOT + (r + 8) * VDIM + (((col >> 3) ^ (4 * (((r + 8) / VRP) % (VC / 4)))) * 8) + (col & 7)];
                const at_u2 x = __builtin_bit_cast(at_u2, __builtin_amdgcn_ds_read_tr16_b64_v4f16((__attribute__((address_space(3))) at_h4*)(v0)));
                const at_u2 y = __builtin_bit_cast(at_u2, __builtin_amdgcn_ds_read_tr16_b64_v4f16((__attribute__((address_space(3))) at_h4*)(v1)));
                vf[d] = __builtin_bit_cast(at_b8, at_u4{x.x, x.y, y.x, y.y});
            }
#pragma unroll
            for (int d = 0; d < DB; d++) acc[d] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(vf[d], __builtin_bit_cast(at_b8, pl), acc[d], 0, 0, 0);
#pragma unroll
            for (int d = 0; d < DB; d++) acc[d] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(vf[d], __builtin_bit_cast(at_b8, pm), acc[d], 0, 0, 0);
#pragma unroll
            for (int d = 0; d < DB; d++) acc[d] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(vf[d], __builtin_bit_cast(at_b8, ph), acc[d], 0, 0, 0);
        }
    }
    // ---- an unsplit launch adds the sink and writes the output, a split one leaves (maximum, denominator, sums)
    l += at_other_half(l, h);
    if (!rv) return;
    const int t = t0 + tq;
    if (a.nsplit > 1) {
        const size_t slot = ((size_t)t * a.heads + head) * a.nsplit + sp;
#pragma unroll
        for (int d = 0; d < DB; d++)
#pragma unroll
            for (int i = 0; i < 16; i += 4)
                *reinterpret_cast<float4*>(&a.part_acc[slot * VDIM + 32 * d + 2 * i + 4 * h]) = make_float4(acc[d][i], acc[d][i + 1], acc[d][i + 2], acc[d][i + 3]);
        if (h == 0) { a.part_ml[slot * 2] = m; a.part_ml[slot * 2 + 1] = l; }
        return;
    }
    float f = 1.0f;
    if (a.sink) {
        const float sk = a.sink[head] * AT_LOG2E, mr = fmaxf(m, sk);
        f = m == -INFINITY ? 0.0f : exp2f(m - mr);
        l = l * f + exp2f(sk - mr);
    }
    f = f / l * (a.out_scale != 0.0f ? a.out_scale : 1.0f);
    const float* gate = a.out_gate ? a.out_gate + (size_t)t * a.ld_gate + (a.gate_elem ? (size_t)head * VDIM : (size_t)head) : nullptr;
    if (gate && !a.gate_elem) f *= 1.0f / (1.0f + expf(-gate[0]));
    uint16_t* o = (uint16_t*)a.out + (size_t)t * (a.out_ld ? a.out_ld : a.heads * VDIM) + (size_t)head * VDIM;
#pragma unroll
    for (int d = 0; d < DB; d++)
#pragma unroll
        for (int i = 0; i < 16; i += 4) {
            const int col = 32 * d + 2 * i + 4 * h;
            uint16_t w[4];
#pragma unroll
            for (int j = 0; j < 4; j++) w[j] = kr_f32_to_bf16(acc[d][i + j] * f * (gate && a.gate_elem ? 1.0f / (1.0f + expf(-gate[col + j])) : 1.0f));
            if (((uintptr_t)(o + col) & 7) == 0) *reinterpret_cast<uint2*>(o + col) = make_uint2(w[0] | ((uint32_t)w[1] << 16), w[2] | ((uint32_t)w[3] << 16));
            else { o[col] = w[0]; o[col + 1] = w[1]; o[col + 2] = w[2]; o[col + 3] = w[3]; }
        }
}

template <int DIM, int VDIM>
__global__ void __launch_bounds__(512, 2) sv_attn_step_kernel(const KrSvAttn a) {
    extern __shared__ __attribute__((aligned(16))) float lds[];
    as_token<DIM, VDIM, 8>(a, blockIdx.x, blockIdx.y, blockIdx.z, lds);
}

template <int DIM, int VDIM> void as_launch(const KrSvAttn& a, hipStream_t st) {
    const int R = a.heads / a.kv_heads, lds = as_lds_bytes(R, VDIM, 8);
    if (kr_lds_optin((const void*)sv_attn_step_kernel<DIM, VDIM>, lds)) return;        // (the step ends with the runtime's error)
    hipLaunchKernelGGL((sv_attn_step_kernel<DIM, VDIM>), dim3(a.T, a.kv_heads, (R + 15) / 16 * a.nsplit), dim3(512), lds, st, a);
}
template <int DIM, int VDIM> void at_launch(const KrSvAttn& a, hipStream_t st) {
    const int TQ = AT_ROWS / (a.heads / a.kv_heads);
    hipLaunchKernelGGL((sv_attn_prompt_kernel<DIM, VDIM>), dim3((a.T - a.n_few) / TQ + a.n_entries, a.kv_heads, a.nsplit), dim3(256), 0, st, a);
}
}  // namespace

bool kr_sv_attn_prompt_fits(int heads, int kv_heads, int dim, int vdim, int ldk, int ldv, int ldq, bool f32) {
    if (f32 || AT_ROWS % (heads / kv_heads) != 0 || ldk % 8 != 0 || ldv % 8 != 0 || ldq % 4 != 0) return false;
    return (dim == 32 || dim == 64 || dim == 128) && (vdim == 32 || vdim == 64 || vdim == 128);
}

// key splits of a launch: workgroups of 128 rows for about two rounds of the chip, four tiles of keys each at least
int kr_sv_attn_prompt_splits(int T, int n_entries, int heads, int kv_heads, int max_visible) {
    const long blocks = (long)(T / (AT_ROWS / (heads / kv_heads)) + n_entries) * kv_heads;
    const int tiles = (max_visible + AT_KEYS - 1) / AT_KEYS;
    long ns = 512 / (blocks > 0 ? blocks : 1);
    if (ns > tiles / 4) ns = tiles / 4;
    return ns < 1 ? 1 : (int)ns;
}

void kr_sv_attn_prompt(const KrSvAttn& a, hipStream_t st) {
#define AT_D(DIM_) do { if (a.vdim == 32) at_launch<DIM_, 32>(a, st); else if (a.vdim == 64) at_launch<DIM_, 64>(a, st); else at_launch<DIM_, 128>(a, st); } while (0)
    if (a.dim == 32) AT_D(32); else if (a.dim == 64) AT_D(64); else AT_D(128);
#undef AT_D
}

bool kr_sv_attn_step_fits(int dim, int vdim, int ldk, int ldv, int ldq, int page_tokens, bool f32) {
    if (f32 || page_tokens % 32 != 0 || ldk % 8 != 0 || ldv % 8 != 0 || ldq % 4 != 0) return false;
    return (dim == 32 || dim == 64 || dim == 128) && (vdim == 32 || vdim == 64 || vdim == 128);      // 256: the split operands no longer fit the registers
}

// Key splits of a decode step: one workgroup up to 256 keys (one round of its waves), then two, four and eight (powers of two: a new count is a new step to capture), beyond 1024
// shares of 512 keys; never more than two workgroups per compute unit in all, which bounds the partial states too.  (us per step of two layers, 1 / 2 / 4 / 8 / 16 shares: one
// request at 100 keys 248 / 248 / 253 / 252 / 253, at 1024 275 / 268 / 266 / 258 / 258; twelve requests at 1024 333 / 322 / 325 / 320 / 331.  Many requests, shares unbounded / at most
// 1024 / at most 512 workgroups: 64 of 8 / 8 heads at 1100 keys 388 / 298 / 279, 128 of 64 / 4 heads at 1100 627 / 507 / 476, 256 of 16 / 2 heads at 2000 960 / 840 / 844.)
int kr_sv_attn_step_splits(int T, int heads, int kv_heads, int max_visible) {
    const long most = std::max(1L, 512 / std::max(1L, (long)T * kv_heads * ((heads / kv_heads + 15) / 16)));
    return (int)std::min(most, (long)(max_visible <= 256 ? 1 : max_visible < 512 ? 2 : max_visible < 1024 ? 4 : std::max(8, max_visible / 512)));
}

void kr_sv_attn_step(const KrSvAttn& a, hipStream_t st) {
#define AS_D(DIM_) do { if (a.vdim == 32) as_launch<DIM_, 32>(a, st); else if (a.vdim == 64) as_launch<DIM_, 64>(a, st); else as_launch<DIM_, 128>(a, st); } while (0)
    if (a.dim == 32) AS_D(32); else if (a.dim == 64) AS_D(64); else AS_D(128);
#undef AS_D
}
