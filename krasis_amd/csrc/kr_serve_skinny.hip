// kr_serve_skinny.hip -- C[M, N] = A[M, K] x W[N, K]^T for few rows of A (decode steps, short prompts) in a bf16 store, on v_mfma_f32_16x16x32_bf16.
//
// Bound: the weight stream (2 N K bytes); the products are free on the matrix cores.  A workgroup owns 16 columns and ALL rows, so a weight byte is read once whatever
// M is; its waves take equal parts of K and meet in LDS (a wave-per-column form has to add 64 lanes per column and re-reads the weights for every eight rows).  The
// strip a wave needs is requested eight steps of 32 k at a time before its first product: with 128 - 2048 workgroups of 64 KB that is what keeps enough bytes in
// flight, LDS staging would only add a hop.  Weights are the first operand (16 columns x 32 k, lane = column + 16 (k / 8)), rows of A the second; rows past M repeat
// the last one (same address, no traffic) and are not stored.
// ACT: A is the gated activation of act_gu, formed once per workgroup into LDS while the first weights travel (the wave-per-column form forms it again per column).
// Grouped problems (one matrix per expert): a strip per problem row; the first row of a group takes the group's rows, the others leave at once.
// Measured, us, before -> now (weights colder than the last cache): 12 rows: 4224 x 2048 23.9 -> 9.4, 2048 x 2048 19.2 -> 5.9, 32768 x 2048 110 -> 33.6 (4.0 TB/s); 1 row:
// 9.3 -> 7.2, 6.6 -> 5.0, 45.6 -> 25.6 (5.2 TB/s); 64 experts of 1536 x 2048, 72 rows 54 -> 46 (5.9 TB/s), 180 rows 92 -> 68.
#include <algorithm>

#include "kr_lds_optin.h"
#include "kr_serve_gemm_dev.h"

namespace {
typedef float sk_f4 __attribute__((ext_vector_type(4)));

template <int MB, int NB, int WV, bool ACT>               // row blocks of 16, column blocks of 16, waves
__device__ __forceinline__ void sk_strip(const KrSvGemm& g, const int by) {      // by: problem row of a grouped problem
    constexpr int U = NB * MB <= 2 ? 8 : 4;                   // k steps requested together
    constexpr int TR = MB * NB < 4 ? MB * NB : 4;             // output tiles per round of the reduction
    __shared__ __attribute__((aligned(16))) float red[WV][TR][256];
    extern __shared__ __attribute__((aligned(16))) uint16_t act[];      // ACT: the rows' activation [16 MB][K + 8]
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, r = lane & 15, q = lane >> 4, n0 = blockIdx.x * 16 * NB;
    int lo = 0, hi = g.M, N = g.N;
    const uint16_t* W = (const uint16_t*)g.W;
    if (g.row_group) {
        const int group = g.row_group[by];
        lo = g.seg[group];
        if (lo != by) return;
        hi = g.seg[group + 1];
        W += (size_t)group * g.w_stride; N = gm_cols(g, group);
    }
    if (n0 >= N) return;
    const int ks = g.K / 32, s0 = ks * wave / WV, s1 = ks * (wave + 1) / WV, lda = g.K + 8;
    const uint16_t* wp[NB];
#pragma unroll
    for (int b = 0; b < NB; b++) wp[b] = W + (size_t)min(n0 + b * 16 + r, N - 1) * g.K + q * 8;
    auto request = [&](gu4 (&wv)[U][NB], int s) {
#pragma unroll
        for (int u = 0; u < U; u++) {
            const int k = min(s + u, s1 - 1) * 32;             // steps past the wave's last one are requested again and not multiplied
#pragma unroll
            for (int b = 0; b < NB; b++) wv[u][b] = *reinterpret_cast<const gu4*>(wp[b] + k);
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
        for (int s = s0; s < s1; s += U) {
            if (!ACT || s > s0) request(wv, s);
            gu4 av[U][MB];
#pragma unroll
            for (int u = 0; u < U; u++) {
                const int k = min(s + u, s1 - 1) * 32;
#pragma unroll
                for (int a = 0; a < MB; a++) av[u][a] = *reinterpret_cast<const gu4*>(ap[a] + k);
            }
#pragma unroll
            for (int u = 0; u < U; u++) {
                if (s + u < s1) {
#pragma unroll
                    for (int a = 0; a < MB; a++)
#pragma unroll
                        for (int b = 0; b < NB; b++) acc[a][b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(gb8, wv[u][b]), __builtin_bit_cast(gb8, av[u][a]), acc[a][b], 0, 0, 0);
                }
            }
        }
        // the waves' partial sums meet, TR tiles of 16 x 16 at a time: tile element (row r, column c) at r * 16 + c, a lane holds four columns of one row
#pragma unroll
        for (int t0 = 0; t0 < MB * NB; t0 += TR) {
            if (t0 > 0) __syncthreads();
#pragma unroll
            for (int t = 0; t < TR; t++) {
                const sk_f4 v = acc[(t0 + t) / NB][(t0 + t) % NB];
                *reinterpret_cast<float4*>(&red[wave][t][r * 16 + q * 4]) = make_float4(v[0], v[1], v[2], v[3]);
            }
            __syncthreads();
            for (int i = tid; i < TR * 256; i += 64 * WV) {
                const int t = i >> 8, e = i & 255, m = m0 + ((t0 + t) / NB) * 16 + (e >> 4), n = n0 + ((t0 + t) % NB) * 16 + (e & 15);
                if (m >= hi || n >= N) continue;
                float v = red[0][t][e];
#pragma unroll
                for (int w = 1; w < WV; w++) v += red[w][t][e];
                gm_store<true>(g, m, n, v);
            }
        }
        if (m0 + 16 * MB < hi) __syncthreads();
    }
}

template <int MB, int NB, int WV, bool ACT>
__global__ void __launch_bounds__(64 * WV) sv_skinny_kernel(const KrSvGemm g) { sk_strip<MB, NB, WV, ACT>(g, blockIdx.y); }
// the experts' and the shared expert's down projection of a step in one launch, both with the activation inside: neither fills the chip, and a launch with its gap costs more
// than the smaller of the two (six expert rows and one row, 2048 x 768: 8.1 + 6.3 -> 8.7 us)
__global__ void __launch_bounds__(256) sv_skinny_pair_kernel(const KrSvGemm e, const KrSvGemm o) {
    if (blockIdx.y == 0) sk_strip<1, 1, 4, true>(o, 0); else sk_strip<1, 1, 4, true>(e, blockIdx.y - 1);
}

int sk_act_lds(const KrSvGemm& g) { return (g.row_group ? 16 : std::min(16, g.M)) * (g.K + 8) * 2; }      // one block of sixteen rows

template <int MB, int NB, int WV>
void sk_launch(const KrSvGemm& g, hipStream_t st) {
    const dim3 grid((g.N + 16 * NB - 1) / (16 * NB), g.row_group ? g.M : 1);
    if (g.act_gu) {
        const int rows = g.row_group ? 16 * MB : std::min(16 * MB, g.M), lds = rows * (g.K + 8) * 2;
        if (kr_lds_optin((const void*)sv_skinny_kernel<MB, NB, WV, true>, lds)) return;
        hipLaunchKernelGGL((sv_skinny_kernel<MB, NB, WV, true>), grid, dim3(64 * WV), lds, st, g);
    } else hipLaunchKernelGGL((sv_skinny_kernel<MB, NB, WV, false>), grid, dim3(64 * WV), 0, st, g);
}
}  // namespace

bool kr_sv_gemm_skinny_fits(const KrSvGemm& g) {
    if (g.K % 32 != 0 || (uintptr_t)g.W % 16 != 0 || g.w_stride % 8 != 0) return false;
    if (g.seg && !g.row_group) return false;
    if (g.act_gu && (g.act_ld % 4 != 0 || (uintptr_t)g.act_gu % 16 != 0)) return false;
    return g.A == nullptr || (g.lda % 8 == 0 && (uintptr_t)g.A % 16 == 0);
}

// The activation inside the launch is formed by every workgroup again: cheaper than a launch of its own (4 - 5 us) up to 16 K values (one matrix; 2048 x 768: 1 row 4.6,
// 12 rows 8.2 us, wave-per-column form 8.0 / 42; 2048 x 6144: 1 row 10.9, 4 rows already 18.6) and, with one matrix per expert, up to 48 rows (24 rows 18.9 us).  Its rows
// have to fit the LDS of two workgroups.
bool kr_sv_gemm_skinny_acts(const KrSvGemm& g) { return g.seg ? g.M <= 48 && g.K <= 1536 : g.M <= 16 && (long)g.M * g.K <= 16384; }

void kr_sv_gemm_skinny(const KrSvGemm& g, hipStream_t st) {
    KrSvGemm p = g;
    if (!g.seg) p.row_group = nullptr;
    // waves: four where the columns alone give every compute unit a workgroup (32768 x 2048, 12 rows: 33.6 us, eight waves 36.4), else eight, which halve a wave's
    // chain of requests (2048 x 768 with the activation, 12 rows: 8.2 us, four waves 9.7)
    if (g.seg || (g.M <= 16 && g.N >= 4096)) sk_launch<1, 1, 4>(p, st);
    else if (g.M <= 16) sk_launch<1, 1, 8>(p, st);
    else sk_launch<2, 1, 8>(p, st);
}

void kr_sv_gemm_skinny_pair(const KrSvGemm& e, const KrSvGemm& o, hipStream_t st) {
    KrSvGemm p = o;
    p.row_group = nullptr;
    const int lds = std::max(sk_act_lds(e), sk_act_lds(p));
    if (kr_lds_optin((const void*)sv_skinny_pair_kernel, lds)) return;
    hipLaunchKernelGGL(sv_skinny_pair_kernel, dim3((std::max(e.N, o.N) + 15) / 16, e.M + 1), dim3(256), lds, st, e, p);
}
