// kr_serve_skinny.hip -- C[M, N] = A[M, K] x W[N, K]^T for few rows of A (decode steps, short prompts) in a bf16 store, on v_mfma_f32_16x16x32_bf16.
//
// Bound: the weight stream (2 N K bytes); the products are free on the matrix cores.  A workgroup owns 16 columns and ALL rows, so a weight byte is read once whatever
// M is; its waves take equal parts of K and meet in LDS (a wave-per-column form has to add 64 lanes per column and re-reads the weights for every eight rows).  The
// strip a wave needs is requested eight steps of 32 k at a time before its first product: with 128 - 2048 workgroups of 64 KB that is what keeps enough bytes in
// flight, LDS staging would only add a hop.  Weights are the first operand (16 columns x 32 k, lane = column + 16 (k / 8)), rows of A the second; rows past M repeat
// the last one (same address, no traffic) and are not stored.
// ACT: A is the gated activation of act_gu, formed once per workgroup into LDS while the first weights travel (the wave-per-column form forms it again per column).
// Grouped problems (one matrix per expert): a strip per problem row; the first row of a group takes the group's rows, the others leave at once.
// Measured, us, before -> now (weights colder than the last cache): 12 rows: 4224 x 2048 23.9 -> 9.3, 2048 x 2048 19.2 -> 5.7, 32768 x 2048 110 -> 33.6 (4.0 TB/s); 1 row:
// 9.3 -> 7.3, 6.6 -> 4.9, 45.6 -> 25.6 (5.2 TB/s); 64 experts of 1536 x 2048, 72 rows 54 -> 46 (5.9 TB/s), 180 rows 92 -> 68.
#include <algorithm>

#include "kr_lds_optin.h"
#include "kr_serve_strip_dev.h"

namespace {
template <int MB, int NB, int WV, bool ACT, int U, bool LINES>
__global__ void __launch_bounds__(64 * WV) sv_skinny_kernel(const KrSvGemm g) {
    __shared__ __attribute__((aligned(16))) float red[sk_red_floats(MB, NB, WV)];
    extern __shared__ __attribute__((aligned(16))) uint16_t act[];
    sk_strip<MB, NB, WV, ACT, false, U, LINES>(g, blockIdx.x, blockIdx.y, red, act);
}
// the experts' and the shared expert's down projection of a step in one launch, both with the activation inside: neither fills the chip, and a launch with its gap costs more
// than the smaller of the two (six expert rows and one row, 2048 x 768: 8.1 + 6.3 -> 8.7 us)
template <int U>
__global__ void __launch_bounds__(256) sv_skinny_pair_kernel(const KrSvGemm e, const KrSvGemm o) {
    __shared__ __attribute__((aligned(16))) float red[sk_red_floats(1, 1, 4)];
    extern __shared__ __attribute__((aligned(16))) uint16_t act[];
    if (blockIdx.y == 0) sk_strip<1, 1, 4, true, false, U>(o, blockIdx.x, 0, red, act); else sk_strip<1, 1, 4, true, false, U>(e, blockIdx.x, blockIdx.y - 1, red, act);
}

// Up to three products of the same rows in one launch, the last one the gate | up pairs of a feed-forward that leave as their activation.  A launch with its gap
// costs what 25 MB of weights cost, and the activation formed in the down projection is formed again by every one of its workgroups.  Two rows, width 2048, feed-forward 6144:
// gate | up and the residual gate behind them, 14336 columns, 13.8 -> 13.9 us, the down projection that no longer forms the activation 15.4 -> 11.4; mixer projections and
// residual gate 2048 x 2048 13.8 + 5.4 -> 13.9 us.
__global__ void __launch_bounds__(256) sv_strips_kernel(const KrSvGemm a, const KrSvGemm b, const KrSvGemm c, const int na, const int nb) {
    __shared__ __attribute__((aligned(16))) float red[sk_red_floats(1, 2, 4)];
    int i = blockIdx.x;
    if (i < na) { sk_strip<1, 1, 4, false, false, 8, true>(a, i, 0, red, nullptr); return; }
    i -= na;
    if (i < nb) { sk_strip<1, 1, 4, false, false, 8, true>(b, i, 0, red, nullptr); return; }
    i -= nb;
    sk_strip<1, 2, 4, false, true, 8, true>(c, i, 0, red, nullptr);
}

int sk_act_lds(const KrSvGemm& g) { return (g.row_group ? 16 : std::min(16, g.M)) * (g.K + 8) * 2; }      // one block of sixteen rows

template <int MB, int NB, int WV, int U, bool LINES>
void sk_launch_u(const KrSvGemm& g, hipStream_t st) {
    const dim3 grid((g.N + 16 * NB - 1) / (16 * NB), g.row_group ? g.M : 1);
    if (g.act_gu) {
        const int rows = g.row_group ? 16 * MB : std::min(16 * MB, g.M), lds = rows * (g.K + 8) * 2;
        if (kr_lds_optin((const void*)sv_skinny_kernel<MB, NB, WV, true, U, LINES>, lds)) return;
        hipLaunchKernelGGL((sv_skinny_kernel<MB, NB, WV, true, U, LINES>), grid, dim3(64 * WV), lds, st, g);
    } else if (g.c_host && g.M > 2) hipLaunchKernelGGL((sv_skinny_kernel<MB, NB, WV, false, U, false>), grid, dim3(64 * WV), 0, st, g);
    else hipLaunchKernelGGL((sv_skinny_kernel<MB, NB, WV, false, U, LINES>), grid, dim3(64 * WV), 0, st, g);
}
template <int MB, int NB, int WV, bool LINES>
void sk_launch(const KrSvGemm& g, hipStream_t st) {
    switch (sk_steps(g.K, WV)) {
        case 4: sk_launch_u<MB, NB, WV, 4, LINES>(g, st); break;
        case 6: sk_launch_u<MB, NB, WV, 6, LINES>(g, st); break;
        default: sk_launch_u<MB, NB, WV, 8, LINES>(g, st); break;
    }
}
template <int U> void sk_pair_launch(const KrSvGemm& e, const KrSvGemm& o, int lds, hipStream_t st) {
    if (kr_lds_optin((const void*)sv_skinny_pair_kernel<U>, lds)) return;
    hipLaunchKernelGGL(sv_skinny_pair_kernel<U>, dim3((std::max(e.N, o.N) + 15) / 16, e.M + 1), dim3(256), lds, st, e, o);
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
    if (g.seg) sk_launch<1, 1, 4, false>(p, st);
    else if (g.M <= 16 && g.N >= 4096) sk_launch<1, 1, 4, true>(p, st);
    else if (g.M <= 16) sk_launch<1, 1, 8, true>(p, st);
    else sk_launch<2, 1, 8, false>(p, st);
}

void kr_sv_gemm_skinny_pair(const KrSvGemm& e, const KrSvGemm& o, hipStream_t st) {
    KrSvGemm p = o;
    p.row_group = nullptr;
    const int lds = std::max(sk_act_lds(e), sk_act_lds(p));
    switch (sk_steps(e.K, 4)) {
        case 4: sk_pair_launch<4>(e, p, lds, st); break;
        case 6: sk_pair_launch<6>(e, p, lds, st); break;
        default: sk_pair_launch<8>(e, p, lds, st); break;
    }
}

bool kr_sv_strips_fits(const KrSvGemm& g) { return g.M > 0 && g.M <= 16 && !g.seg && !g.act_gu && !g.c_rows && !g.c_host && kr_sv_gemm_skinny_fits(g); }

void kr_sv_strips(const KrSvGemm& a, const KrSvGemm& b, const KrSvGemm& c, hipStream_t st) {
    KrSvGemm p[3] = {a, b, c};
    int n[3];
    for (int i = 0; i < 3; i++) { p[i].row_group = nullptr; n[i] = p[i].M <= 0 ? 0 : ((i == 2 ? p[i].glu_f : p[i].N) + 15) / 16; }
    if (n[0] + n[1] + n[2] > 0) hipLaunchKernelGGL(sv_strips_kernel, dim3(n[0] + n[1] + n[2]), dim3(256), 0, st, p[0], p[1], p[2], n[0], n[1]);
}
