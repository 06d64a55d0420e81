// kr_serve_step.hip -- decode steps of a parallel block with experts (bf16): the two branches of the block, attention and feed-forward, share their launches.
//
// A layer of such a step is a chain of launches that each move 8 - 40 MB (2 - 8 us of memory time) or nothing worth counting, and a launch that depends on the one before it
// costs 4 - 5 us whatever it does.  The branches do not depend on one another until the residual sum, so they go side by side:
//   attention of every token            |  experts' gate and up product, the activation formed from its sums    (sv_attn_up_kernel)
//   attention's output projection       |  experts' down projection  |  the shared expert's                     (sv_downs_kernel)
// A workgroup's number says which part it is; attention, whose chain is the longest, comes first.  A side stream instead was no gain: its two joins cost what the overlap gives.
// Per layer with the preparation beside the router (kr_serve_ops.hip): eight launches become five,
// 54 -> 39 us with one request (16 / 2 heads of 128, 64 experts of 2048 x 768, top 6), eleven become five, 143 -> 113 us with twelve.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <algorithm>

#include "kr_lds_optin.h"
#include "kr_serve_attn_dev.h"
#include "kr_serve_strip_dev.h"

namespace {
// Eight waves of at most 128 registers (the lean form of attention), two workgroups to a compute unit, for what streams the experts beside it.
constexpr int AU_WAVES = 8;
// Up to this many problem rows each is taken alone, a wave per gate column and its up column: whole matrix rows per request and no wait for the group's
// bounds.  A step, us, rows alone / strips of 16 + 16 columns: 24 rows on 64 experts of 2 x 768 x 2048, two layers, 192 / 206, on 128 of 2 x 1536 x 4096, one layer, 291 / 311.
// With more rows than experts an expert's matrix is read by several rows, which costs little while all of them stay in the 256 MB cache (two layers: 18 rows on 16 experts of 2 x 768 x 2048 167 / 178,
// 24 on 8 168 / 164) and much beyond it (one layer of 8 of 2 x 4096 x 4096, 537 MB: 12 rows 289 / 268, 24 rows 414 / 300): hence half of it.
constexpr int AU_ROWS = 24;
bool au_rows_alone(const KrSvGemm& up) { return up.M <= AU_ROWS && (up.M <= up.n_groups || (size_t)up.n_groups * up.w_stride * 2 <= (size_t)128 << 20); }
template <int DIM, int VDIM>
__global__ void __launch_bounds__(64 * AU_WAVES, 4) sv_attn_up_kernel(const KrSvAttn a, const KrSvGemm up, const int n_attn, const int strips, const int alone) {
    extern __shared__ __attribute__((aligned(16))) float lds[];
    // (quotients are formed on the vector unit; without readfirstlane all that follows from them would stay there)
    if ((int)blockIdx.x < n_attn) {
        const int th = __builtin_amdgcn_readfirstlane(blockIdx.x / a.T), bz = __builtin_amdgcn_readfirstlane(th / a.kv_heads);
        as_token<DIM, VDIM, AU_WAVES, true>(a, blockIdx.x - th * a.T, th - bz * a.kv_heads, bz, lds);
    } else {
        const int i = blockIdx.x - n_attn, by = __builtin_amdgcn_readfirstlane(i / strips);
        if (alone) sk_row_glu<AU_WAVES>(up, i - by * strips, by, a.T == 1);
        else sk_strip<1, 2, AU_WAVES, false, true>(up, i - by * strips, by, lds, nullptr);
    }
}

// U: k steps together of the down projections, by their K (sk_steps); attention's projection takes eight.  128 registers for the requests of half lines: without the bound, or with one for more waves
// to a SIMD, the compiler orders them worse (72 rows on 43 of 64 experts of 2048 x 768 27.0 us, 29.1 without); whole lines are as quick without it.
// LINES: how the weights are read (sk_strip), whole lines up to sixteen expert rows (us, halves / lines: 16 rows on 16 of 128 experts of 4096 x 1536 44.1 / 38.9, 12 on 11 of 64 of 2048 x 768
// 10.9 / 10.2, of 2048 x 704 11.1 / 10.9).  Beyond it depends: 24 rows of 4096 x 1536 59.7 / 53.5, 96 161 / 154, but 72 of 2048 x 768 27.0 / 27.8, of 2048 x 704 27.5 / 30.1.
template <int U, bool LINES>
__global__ void __launch_bounds__(256, LINES ? 1 : 4) sv_downs_kernel(const KrSvGemm o, const KrSvGemm e, const KrSvGemm sh, const int so, const int ss, const int se) {
    __shared__ __attribute__((aligned(16))) float red[sk_red_floats(1, 1, 4)];
    extern __shared__ __attribute__((aligned(16))) uint16_t act[];
    int i = blockIdx.x;
    if (i < so) { sk_strip<1, 1, 4, false, false, 8, LINES>(o, i, 0, red, act); return; }
    i -= so;
    if (i < ss) { sk_strip<1, 1, 4, true, false, U, LINES>(sh, i, 0, red, act); return; }
    i -= ss;
    const int by = __builtin_amdgcn_readfirstlane(i / se);
    sk_strip<1, 1, 4, false, false, U, LINES>(e, i - by * se, by, red, act);
}
template <int U, bool LINES> void downs_launch_u(const KrSvGemm& o, const KrSvGemm& e, const KrSvGemm& sh, int so, int ss, int se, int lds, hipStream_t st) {
    if (kr_lds_optin((const void*)sv_downs_kernel<U, LINES>, lds)) return;
    hipLaunchKernelGGL((sv_downs_kernel<U, LINES>), dim3(so + ss + se * e.M), dim3(256), lds, st, o, e, sh, so, ss, se);
}
template <int U> void downs_launch(const KrSvGemm& o, const KrSvGemm& e, const KrSvGemm& sh, int so, int ss, int se, int lds, hipStream_t st) {
    if (e.M <= 16) downs_launch_u<U, true>(o, e, sh, so, ss, se, lds, st); else downs_launch_u<U, false>(o, e, sh, so, ss, se, lds, st);
}

template <int DIM, int VDIM> void au_launch(const KrSvAttn& a, const KrSvGemm& up, hipStream_t st) {
    const int R = a.heads / a.kv_heads, lds = std::max({as_lds_bytes(R, VDIM, AU_WAVES), as_lean_lds_bytes(DIM), sk_red_floats(1, 2, AU_WAVES) * (int)sizeof(float)});
    const int n_attn = a.T * a.kv_heads * ((R + 15) / 16) * a.nsplit, alone = au_rows_alone(up), cols = alone ? AU_WAVES : 16, strips = (up.glu_f + cols - 1) / cols;
    if (kr_lds_optin((const void*)sv_attn_up_kernel<DIM, VDIM>, lds)) return;        // (the step ends with the runtime's error)
    hipLaunchKernelGGL((sv_attn_up_kernel<DIM, VDIM>), dim3(n_attn + strips * up.M), dim3(64 * AU_WAVES), lds, st, a, up, n_attn, strips, alone);
}
}  // namespace

// shapes: whole fragments for every product, a choice that one workgroup of kr_sv_prep_route makes, and experts with few enough rows that a strip per expert reads its weights about once
// (the rule of the strips alone, kr_serve_gemm.hip)
bool kr_sv_step_join_fits(int T, int width, int o_cols, int experts, int top, int groups, int ff) {
    return T <= 16 && width % 32 == 0 && o_cols % 32 == 0 && ff % 32 == 0 && experts <= 128 && top <= 64 && groups <= 64 && T * top <= 8 * experts;
}

// Beside the experts' product attention only has to be no longer than that: a workgroup takes 256 keys in 1.5 us past its first few us, the product min(T top, experts)
// matrices at some 5 TB/s.  One workgroup per token and key head while that covers the keys (no merge of partial states then), else powers of two, never more than alone.
// (A step of two layers without a window, us, launches of their own / joined, 64 experts of 2 x 768 x 2048: one request at 4000 keys 240 / 175, 16000 254 / 187, 40000 274 / 200; four at 8000 352 / 325;
// twelve at 2500 506 / 446; two at 8000 with 16 / 16 heads 322 / 256; 128 experts of 2 x 1536 x 4096, one at 16000 458 / 434.)
int kr_sv_step_join_splits(int T, int heads, int kv_heads, int max_visible, int width, int ff, int experts, int top) {
    const int alone = kr_sv_attn_step_splits(T, heads, kv_heads, max_visible);
    const double up_us = (double)std::min(T * top, experts) * 4.0 * ff * width / 5e6;
    const long keys = 256 * std::max(1L, (long)((up_us - 3.0) / 1.5));
    int n = 1;
    while (n < alone && (long)n * keys < max_visible) n *= 2;
    return std::min(n, alone);
}

void kr_sv_attn_up(const KrSvAttn& a, const KrSvGemm& up, hipStream_t st) {
#define AU_D(DIM_) do { if (a.vdim == 32) au_launch<DIM_, 32>(a, up, st); else if (a.vdim == 64) au_launch<DIM_, 64>(a, up, st); else au_launch<DIM_, 128>(a, up, st); } while (0)
    if (a.dim == 32) AU_D(32); else if (a.dim == 64) AU_D(64); else AU_D(128);
#undef AU_D
}

// sh: the shared expert's down projection with its activation inside (act_gu), or M = 0
void kr_sv_downs(const KrSvGemm& o, const KrSvGemm& e, const KrSvGemm& sh, hipStream_t st) {
    const int so = (o.N + 15) / 16, ss = sh.M > 0 ? (sh.N + 15) / 16 : 0, se = (e.N + 15) / 16;
    const int lds = sh.M > 0 ? std::min(16, sh.M) * (sh.K + 8) * 2 : 0;
    KrSvGemm ov = o, sv = sh;
    ov.row_group = nullptr; sv.row_group = nullptr;
    switch (sk_steps(e.K, 4)) {
        case 4: downs_launch<4>(ov, e, sv, so, ss, se, lds, st); break;
        case 6: downs_launch<6>(ov, e, sv, so, ss, se, lds, st); break;
        default: downs_launch<8>(ov, e, sv, so, ss, se, lds, st); break;
    }
}
