// kr_serve_strip_dev.h -- a workgroup's strip of columns of C[M, N] = A[M, K] x W[N, K]^T for few rows, bf16 (kr_serve_skinny.hip has the reasons), shared by the
// launches of one product and the launches that put several products, or a product and attention, side by side (kr_serve_step.hip).
#ifndef KR_SERVE_STRIP_DEV_H
#define KR_SERVE_STRIP_DEV_H
#include <type_traits>

#include "kr_serve_gemm_dev.h"

typedef float sk_f4 __attribute__((ext_vector_type(4)));

constexpr int sk_red_floats(int MB, int NB, int WV) { return WV * (MB * NB < 4 ? MB * NB : 4) * 256; }

// k steps requested together: the count that leaves the fewest requests of no use behind a wave's last step (they are made all the same, for the last step's bytes again).  Eight where
// six do, with 72 rows on 43 of 64 experts of 2048 x 768, 33.3 us where 26.8 do; 24 on 24 of 128 of 4096 x 1536 65.7 and 59.5.
constexpr int sk_steps(int K, int WV) {
    const int steps = (K / 32 + WV - 1) / WV;
    int best = 8;
    for (int u : {6, 4}) if ((steps + u - 1) / u * u < (steps + best - 1) / best * best) best = u;
    return best;
}
// MB, NB: row and column blocks of 16; WV: waves.  bx: strip, by: problem row of a grouped problem; red: sk_red_floats of LDS, act (with ACT): the rows' activation [16 MB][K + 8].
// GLU (NB = 2): the strip is 16 gate columns, counted from g.glu_lo, and the 16 up columns that belong to them; their activation goes to g.glu_out, nothing to C.
template <int MB, int NB, int WV, bool ACT, bool GLU = false, int U = NB * MB <= 2 ? 8 : 4, bool LINES = false>      // U: k steps requested together; LINES: how (below)
__device__ __forceinline__ void sk_strip(const KrSvGemm& g, const int bx, const int by, float* red, uint16_t* act) {
    static_assert(!GLU || (NB == 2 && MB == 1), "a gate tile and its up tile");
    static_assert(!LINES || U % 2 == 0, "lines are taken by pairs of steps");
    constexpr int TR = MB * NB < 4 ? MB * NB : 4;             // output tiles per round of the reduction
    // (the wave's number is scalar, and so are its k steps: 112 -> 74 registers)
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), r = lane & 15, q = lane >> 4, n0 = bx * 16 * (GLU ? 1 : NB);
    int lo = 0, hi = g.M, N = g.N;
    const uint16_t* W = (const uint16_t*)g.W;
    if (g.row_group) {
        const int group = g.row_group[by];
        lo = g.seg[group];
        if (lo != by) return;
        hi = g.seg[group + 1];
        W += (size_t)group * g.w_stride; N = gm_cols(g, group);
    }
    if (n0 >= (GLU ? g.glu_f : N)) return;
    float* host = gm_host(g.c_host);
    const int ks = g.K / 32, s0 = ks * wave / WV, s1 = ks * (wave + 1) / WV, lda = g.K + 8;
    // How the weights are read: half a line from each of the sixteen columns per request, or (LINES) whole 128-byte lines, two k steps of eight columns (lanes r < 8 the first step, the others the second;
    // the even one of a pair of requests takes columns 0 - 7 of the block, the odd one 8 - 15), which lanes r and r ^ 8 then trade, and past the caches.  Where a wave's part of K begins at an odd step,
    // or K is an odd number of them, a pair holds halves of two lines (12 rows of 2048 x 704, us, halves / lines 4.31 / 3.95, of 3072 x 1056 4.70 / 4.68).  For matrices that a step meets once
    // and whose strips are in flight together (two rows of 2048 x 6144 11.2 / 10.3, 2048 x 2048 5.48 / 4.95, 12 rows of 4224 x 2048 10.5 / 9.4); a matrix that is still in the caches is up to 15 % slower
    // so.  Not for experts whose workgroups come in many rounds (sv_downs_kernel), nor for more than two rows that go to host memory (32768 columns, a step of twelve requests 314 / 333, of three 156 / 160;
    // one and two gain, not there but in the launches of the next step, whose matrices the vocabulary's 134 MB then leave in the last cache).
    const uint16_t* wp[NB][LINES ? 2 : 1];
#pragma unroll
    for (int b = 0; b < NB; b++)
#pragma unroll
        for (int t = 0; t < (LINES ? 2 : 1); t++) {
            const int c = LINES ? 8 * t + (r & 7) : r;
            wp[b][t] = W + (size_t)(GLU ? g.glu_lo + min(n0 + c, g.glu_f - 1) + b * g.glu_f : min(n0 + b * 16 + c, N - 1)) * g.K + q * 8;
        }
    auto request = [&](gu4 (&wv)[U][NB], int s) {
#pragma unroll
        for (int u = 0; u < U; u++) {
            const int k = min(LINES ? s + (u & ~1) + (r >> 3) : s + u, s1 - 1) * 32;      // steps past the wave's last one are requested again and not multiplied
#pragma unroll
            for (int b = 0; b < NB; b++) {
                const gu4* p = reinterpret_cast<const gu4*>(wp[b][LINES ? u & 1 : 0] + k);
                wv[u][b] = LINES ? __builtin_nontemporal_load(p) : *p;
            }
        }
    };
    [[maybe_unused]] auto trade = [&](gu4 (&wv)[U][NB], int u, int b) {         // lanes r and r ^ 8: step u + t of column r in wv[u + t]
#pragma unroll
        for (int e = 0; e < 4; e++) {
            const uint32_t x = wv[u][b][e], y = wv[u + 1][b][e];
            wv[u][b][e] = __builtin_amdgcn_update_dpp(x, y, 0x128, 0xF, 0xC, false);        // row_ror:8
            wv[u + 1][b][e] = __builtin_amdgcn_update_dpp(y, x, 0x128, 0xF, 0x3, false);
        }
    };
    for (int m0 = lo; m0 < hi; m0 += 16 * MB) {
        const uint16_t* ap[MB];
        gu4 wv[U][NB];
        if constexpr (ACT) {
            if (s0 < s1) request(wv, s0);                      // the weights' first strip travels while the activation is formed
            const int rows = min(16 * MB, hi - m0), kv = g.K / 4;
            const int uoff = g.act_kind == KR_SV_ACT_RELU2 || g.up_tab ? 0 : g.K;      // no up columns (un-gated, or taken from a table): the second read repeats the first
            for (int i = tid; i < rows * kv; i += 64 * WV) {
                const int m = i / kv, k = (i - m * kv) * 4, src = g.a_rows ? g.a_rows[m0 + m] : m0 + m;
                const float w = g.act_row_w ? g.act_row_w[m0 + m] : 1.0f;
                const float* gp = g.act_gu + (size_t)src * g.act_ld + k;
                const float4 gg = *reinterpret_cast<const float4*>(gp);
                float4 uu = *reinterpret_cast<const float4*>(gp + uoff);
                if (g.up_tab) {
                    const uint16_t* t = (const uint16_t*)g.up_tab + (size_t)g.up_rows[m0 + m] * g.up_ld + g.up_off + k;
                    uu = make_float4(gm_ld(t), gm_ld(t + 1), gm_ld(t + 2), gm_ld(t + 3));
                }
                const uint32_t x0 = kr_f32_to_bf16(gm_act(gg.x * w, uu.x * w, g.act_kind, g.act_limit, g.act_alpha)), x1 = kr_f32_to_bf16(gm_act(gg.y * w, uu.y * w, g.act_kind, g.act_limit, g.act_alpha));
                const uint32_t x2 = kr_f32_to_bf16(gm_act(gg.z * w, uu.z * w, g.act_kind, g.act_limit, g.act_alpha)), x3 = kr_f32_to_bf16(gm_act(gg.w * w, uu.w * w, g.act_kind, g.act_limit, g.act_alpha));
                *reinterpret_cast<uint2*>(&act[m * lda + k]) = make_uint2(x0 | (x1 << 16), x2 | (x3 << 16));
            }
            __syncthreads();
        }
#pragma unroll
        for (int a = 0; a < MB; a++) {
            const int m = min(m0 + a * 16 + r, hi - 1), src = g.a_rows ? g.a_rows[m] : m;
            ap[a] = ACT ? act + (m - m0) * lda + q * 8 : (const uint16_t*)g.A + (size_t)src * g.lda + q * 8;
        }
        sk_f4 acc[MB][NB];
#pragma unroll
        for (int a = 0; a < MB; a++)
#pragma unroll
            for (int b = 0; b < NB; b++) acc[a][b] = sk_f4{0.0f, 0.0f, 0.0f, 0.0f};
        // U steps of k; part: fewer are left, the others' operands are zeros.  No branch stands around a product: a matrix instruction does not heed the execution mask, and the compiler
        // puts a request that only the product behind a branch needs behind that branch too, a round trip of its own (us, branches / none: 72 rows on 43 of 64 experts of 2048 x 768 31.1 / 27.0,
        // 96 on 71 of 128 of 4096 x 1536 189 / 162, 20 rows of 2048 x 768 5.44 / 4.90).
        auto products = [&](int s, auto part) {
            gu4 av[U][MB];
#pragma unroll
            for (int u = 0; u < U; u++) {
                const int k = min(s + u, s1 - 1) * 32;
#pragma unroll
                for (int a = 0; a < MB; a++) av[u][a] = *reinterpret_cast<const gu4*>(ap[a] + k);
            }
            // every request before the first product (us, without / with: 24 rows on 22 of 64 experts of 2048 x 768 19.1 / 16.4).  Not where registers are short (pairs beside attention: 20 bytes of
            // scratch, twelve requests' step 333 / 338), nor where the rows come from LDS (experts' and shared expert's strips of twelve requests alike 12.9 / 13.5)
            if (!LINES && !ACT && MB * NB == 1 && U > 4) __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int u = 0; u < U; u++) {
                if (LINES && u % 2 == 0) {
#pragma unroll
                    for (int b = 0; b < NB; b++) trade(wv, u, b);
                }
                const bool none = decltype(part)::value && s + u >= s1;
#pragma unroll
                for (int a = 0; a < MB; a++)
#pragma unroll
                    for (int b = 0; b < NB; b++) {
                        const gu4 zero = {0, 0, 0, 0}, x = none ? zero : wv[u][b], y = none ? zero : av[u][a];
                        acc[a][b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(gb8, x), __builtin_bit_cast(gb8, y), acc[a][b], 0, 0, 0);
                    }
            }
        };
        int s = s0;
        for (; s + U <= s1; s += U) {
            if (!ACT || s > s0) request(wv, s);
            products(s, std::false_type{});
        }
        if (s < s1) {
            if (!ACT || s > s0) request(wv, s);
            products(s, std::true_type{});
        }
        // the waves' partial sums meet, TR tiles of 16 x 16 at a time: tile element (row r, column c) at r * 16 + c, a lane holds four columns of one row
#pragma unroll
        for (int t0 = 0; t0 < MB * NB; t0 += TR) {
            if (t0 > 0) __syncthreads();
#pragma unroll
            for (int t = 0; t < TR; t++) {
                const sk_f4 v = acc[(t0 + t) / NB][(t0 + t) % NB];
                *reinterpret_cast<float4*>(&red[(wave * TR + t) * 256 + r * 16 + q * 4]) = make_float4(v[0], v[1], v[2], v[3]);
            }
            __syncthreads();
            if constexpr (GLU) {
                for (int e = tid; e < 256; e += 64 * WV) {
                    const int m = m0 + (e >> 4), n = n0 + (e & 15);
                    if (m >= hi || n >= g.glu_f) continue;
                    float gt = red[e], up = red[256 + e];
#pragma unroll
                    for (int w = 1; w < WV; w++) { gt += red[w * TR * 256 + e]; up += red[(w * TR + 1) * 256 + e]; }
                    if (g.bias) { gt += g.bias[g.glu_lo + n]; up += g.bias[g.glu_lo + g.glu_f + n]; }
                    const float wt = g.glu_row_w ? g.glu_row_w[m] : 1.0f;
                    ((uint16_t*)g.glu_out)[(size_t)m * g.glu_f + n] = kr_f32_to_bf16(gm_act_once(gt * wt, up * wt, g.glu_kind, g.glu_limit, g.glu_alpha));
                }
                continue;
            }
            for (int i = tid; i < TR * 256; i += 64 * WV) {
                const int t = i >> 8, e = i & 255, m = m0 + ((t0 + t) / NB) * 16 + (e >> 4), n = n0 + ((t0 + t) % NB) * 16 + (e & 15);
                if (m >= hi || n >= N) continue;
                float v = red[t * 256 + e];
#pragma unroll
                for (int w = 1; w < WV; w++) v += red[(w * TR + t) * 256 + e];
                gm_store<true>(g, m, n, v, host);
            }
        }
        if (m0 + 16 * MB < hi) __syncthreads();
    }
}

// Column n of the gate and up product of problem row `by`, K over a wave's lanes.  PAST: past the caches.
template <bool PAST>
__device__ __forceinline__ void sk_row_glu_column(const KrSvGemm& g, const int n, const int by, const int group) {
    constexpr int U = 4;                                      // 16-byte pieces of K requested together, of both matrices
    const int lane = threadIdx.x & 63;
    const uint16_t* W = (const uint16_t*)g.W + (size_t)group * g.w_stride + (size_t)n * g.K;
    const uint16_t* A = (const uint16_t*)g.A + (size_t)(g.a_rows ? g.a_rows[by] : by) * g.lda;
    float gt = 0.0f, up = 0.0f;
    for (int k0 = 0; k0 < g.K; k0 += 512 * U) {
        gu4 wg[U], wu[U], av[U];
#pragma unroll
        for (int u = 0; u < U; u++) {
            const int k = min(k0 + 512 * u + lane * 8, g.K - 8);      // lanes past the row's end read its last piece and multiply it by zero
            const gu4 *pg = reinterpret_cast<const gu4*>(W + k), *pu = reinterpret_cast<const gu4*>(W + (size_t)g.glu_f * g.K + k);
            wg[u] = PAST ? __builtin_nontemporal_load(pg) : *pg;
            wu[u] = PAST ? __builtin_nontemporal_load(pu) : *pu;
        }
#pragma unroll
        for (int u = 0; u < U; u++) {
            const int k = k0 + 512 * u + lane * 8;
            av[u] = *reinterpret_cast<const gu4*>(A + min(k, g.K - 8));
            if (k >= g.K) av[u] = gu4{0, 0, 0, 0};
        }
#pragma unroll
        for (int u = 0; u < U; u++)
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const float a0 = __uint_as_float(av[u][i] << 16), a1 = __uint_as_float(av[u][i] & 0xFFFF0000u);
                gt = __builtin_fmaf(a0, __uint_as_float(wg[u][i] << 16), gt); gt = __builtin_fmaf(a1, __uint_as_float(wg[u][i] & 0xFFFF0000u), gt);
                up = __builtin_fmaf(a0, __uint_as_float(wu[u][i] << 16), up); up = __builtin_fmaf(a1, __uint_as_float(wu[u][i] & 0xFFFF0000u), up);
            }
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) { gt += __shfl_xor(gt, o); up += __shfl_xor(up, o); }
    const float wt = g.glu_row_w ? g.glu_row_w[by] : 1.0f;
    if (lane == 0) ((uint16_t*)g.glu_out)[(size_t)by * g.glu_f + n] = kr_f32_to_bf16(gm_act_once(gt * wt, up * wt, g.glu_kind, g.glu_limit, g.glu_alpha));
}
// The gate and up product of problem row `by` alone, columns [WV bx, WV bx + WV) of g.glu_f, one per wave: for few rows, which seldom meet an expert twice.  A wave reads whole
// rows of the matrix and waits for nothing but its row's expert and its neighbours' (rows of one expert stand together).  A row that has its expert to itself reads past the caches;
// where a neighbour reads the matrix too it has to stay (us a step: 24 rows on 8 of 128 experts of
// 2 x 1536 x 4096, one layer, all past the caches / none / this rule 261 / 238 / 239, on 22 of them 301 / 304 / 298; one request, six rows, two layers of 64 of 2 x 768 x 2048 132 / 139 / 131).
// one: the rows of one token, whose experts differ; they do not wait for neighbours (a chat turn 5806 -> 5763).
template <int WV>
__device__ __forceinline__ void sk_row_glu(const KrSvGemm& g, const int bx, const int by, const bool one) {
    const int n = bx * WV + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    if (n >= g.glu_f) return;
    if (one) { sk_row_glu_column<true>(g, n, by, g.row_group[by]); return; }
    const int group = g.row_group[by], before = g.row_group[max(by - 1, 0)], behind = g.row_group[min(by + 1, g.M - 1)];
    if ((before != group || by == 0) && (behind != group || by == g.M - 1)) sk_row_glu_column<true>(g, n, by, group);
    else sk_row_glu_column<false>(g, n, by, group);
}

#endif
