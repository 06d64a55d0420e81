// kr_serve_tile.hip -- C[M, N] = A[M, K] x W[N, K]^T for prompt-sized problems, single matrix or one matrix per expert, of a bf16 store (an f32 store's:
// kr_serve_tile_f32.hip).
//
// Bound: the matrix cores (about 1350 TFLOP/s is what a large library product reaches here; nominal 2500).  Both operands travel from memory to LDS by
// global_load_lds_dwordx4 into a ring of slots of 64 k (no staging registers; whole cache lines), fragments read while products run.  What the large tile buys:
// 256 x 256 by eight waves of 128 x 64 reads 48 KB of fragments per 64 matrix instructions and SIMD and 64 KB of operands per slot; 128 x 128 by four waves of 64 x 64 needs
// a third more of the first and twice the second for the same products, and neither the LDS nor the L2 rate hides behind the matrix cores then.
// What the two larger tiles wait for is the operands: a slot's requests take the CU's 64 bytes a cycle of L1 path for half of the slot's matrix time, and with two whole slots
// in turn they had one slot's time for that and for the way to L2 or memory and back (3300 x 4096 x 8192 in clocks of a CU: matrix instructions alone 287 k, with the
// fragment reads 318 k, with the requests 466 k).  So a slot is given back by parts: the fragments of W's slot and of one row block of A's stand in registers before they
// are multiplied, a part of the ring is free as soon as it has been read, and its next request leaves then, one and a half slots of time ahead of its use (348 k clocks).
// LDS-DMA writes lane-linear (lane i at base + 16 i), so bank conflicts are avoided on the SOURCE side: the 16-byte chunk c of row r sits at
// position c ^ (r / 2 % 8) of its 128-byte row and the fragment reads apply the same map (without it 1.6 - 2.1 x slower).
// Measured, us, slots whole -> by parts: 3300 x 4096 x 8192 238 -> 208 (1064 TFLOP/s), 3300 x 12416 x 4096 363 -> 344, 4096 x 4160 x 2048 101 -> 87, 2500 x 4160 x 2048 66 -> 55,
// 3249 x 2048 x 6144 111 -> 92, 500 x 4160 x 2048 26.3 -> 20.2; 64 experts, 24576 x 1536 x 2048 237 -> 210, x 2048 x 768 133 -> 120 (201 MB of f32 results), 15000 x 1536 x 2048 188 -> 149;
// under lasting load the clock falls and the gains are 7 - 12 %.
#include <algorithm>
#include <cmath>
#include <type_traits>

#include "kr_lds_optin.h"
#include "kr_serve_tile_dev.h"

namespace {
// GLU: columns [glu_lo, glu_lo + 2 glu_f) leave as the gated activation.  Their tiles come behind those of the other columns (the column numbers of those close the gap): half a
// tile of gates and the up columns that belong to them, laid out so that a wave holds both factors of its elements.  The f32 pair is not written and read again and
// the activation's launch is gone: 24576 rows of 2 x 768 on 64 experts, product and activation, 242 + 55 -> 252 us; a 4096-token prompt of four layers 4.06 -> 3.80 ms.
template <int BM, int BN, int WM, int WN, int DEPTH, int WPS, bool GLU>  // WM x WN waves; WPS: waves per SIMD the register budget is for
__global__ void __launch_bounds__(64 * WM * WN, WPS) sv_tile_kernel(const KrSvGemm g) {
    constexpr int MB = BM / (32 * WM), NB = BN / (32 * WN);    // 32 x 32 blocks of a wave
    constexpr int RA = 4 / WN, RW = 4 * NB / WM;               // requests of 8 rows that a wave makes for a row block of A's slot and for W's slot
    constexpr int BK = TL_ROW / 2, CH = 8;                     // k of a slot, elements of a chunk
    constexpr uint32_t AS = BM * TL_ROW, WS = BN * TL_ROW;     // bytes of a slot of A and of W: A's slots come first
    extern __shared__ __attribute__((aligned(1024))) uint8_t ring_[];
    int bx = blockIdx.x, by = blockIdx.y;
    // Workgroups go round the eight XCDs, each with its own L2.  With a column count of a multiple of eight an XCD sees the same columns of W for all rows; otherwise,
    // and with one matrix per expert, it is given whole pairs of row tiles: their rows stay in its L2, the pair shares the columns of W.
    // (4096 x 4224 x 2048: 109 -> 98 us; 64 experts, 24576 x 1536 x 2048: 290 -> 275; but 3250 x 8192 x 2048, 64 columns: 146 as it is, 163 in pairs.)
    if (g.seg || gridDim.x % 8 != 0) {
        const int gx = gridDim.x, L = by * gx + bx, band = L / (16 * gx), rem = L - band * 16 * gx, rows = min(16, (int)gridDim.y - band * 16);
        if (rows == 16) { by = band * 16 + 2 * (rem & 7) + ((rem >> 3) & 1); bx = rem >> 4; }
        else { by = band * 16 + rem % rows; bx = rem / rows; }
    }
    int group = 0, m0 = by * BM, mend = g.M;
    if (g.seg && !gm_find_tile(g.seg, g.n_groups, by, BM, group, m0, mend)) return;
    const int plain = GLU ? g.N - 2 * g.glu_f : 0, plain_tiles = (plain + BN - 1) / BN;      // GLU: columns outside the pairs, and their tiles
    const bool pairs = GLU && bx >= plain_tiles;
    const int n0 = GLU ? (pairs ? (bx - plain_tiles) * (BN / 2) : bx * BN) : bx * BN, N = GLU ? (pairs ? g.glu_f : plain) : gm_cols(g, group);
    if (n0 >= N) return;
    auto column = [&](int n) { return GLU && n >= g.glu_lo ? n + 2 * g.glu_f : n; };         // of C and row of W, of a column outside the pairs
    const uint16_t* A = (const uint16_t*)g.A;
    const uint16_t* W = (const uint16_t*)g.W + (size_t)group * g.w_stride;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), r = lane & 31, h = lane >> 5, wr = wave / WN, wc = wave % WN;
    const uint16_t* as[MB][RA]; const uint16_t* ws[RW];
#pragma unroll
    for (int a = 0; a < MB; a++)
#pragma unroll
        for (int i = 0; i < RA; i++) {
            const int row = a * 32 * WM + (wave * RA + i) * 8 + (lane >> 3), ch = (lane & 7) ^ ((row >> 1) & 7), m = min(m0 + row, mend - 1);
            as[a][i] = A + (size_t)(g.a_rows ? g.a_rows[m] : m) * g.lda + ch * CH;
        }
#pragma unroll
    for (int i = 0; i < RW; i++) {
        const int row = (wave * RW + i) * 8 + (lane >> 3), ch = (lane & 7) ^ ((row >> 1) & 7);
        if (pairs) {                                           // a wave's columns: its gates, then their up factors
            constexpr int WC = BN / WN;
            const int j = n0 + row / WC * (WC / 2) + row % (WC / 2), up = row % WC >= WC / 2;
            ws[i] = W + (size_t)(g.glu_lo + up * g.glu_f + min(j, N - 1)) * g.K + ch * CH;
        } else ws[i] = W + (size_t)column(min(n0 + row, N - 1)) * g.K + ch * CH;
    }
    const uint32_t ringa = __builtin_amdgcn_readfirstlane(tl_lds_addr(ring_)), basea = ringa + wave * RA * 1024u, basew = ringa + DEPTH * AS + wave * RW * 1024u;
    gv16f acc[MB][NB];
#pragma unroll
    for (int a = 0; a < MB; a++)
#pragma unroll
        for (int b = 0; b < NB; b++)
#pragma unroll
            for (int i = 0; i < 16; i++) acc[a][b][i] = 0.0f;
    const int steps = g.K / BK;
    // A tile's row blocks go round the waves' rows (block a of wave row wr: rows 32 (a WM + wr)), so that the last tile of a matrix or an expert, which is seldom full, takes only the
    // blocks it has: the k loop exists once per number of them, and rows past the last block are not requested.  24576 rows on 64 experts, about 384 each, 2 x 768 x 2048: 235 -> 222 us; 27500
    // rows on 128, 2 x 1536 x 4096: 730 -> 702, and x 4096 x 1536 308 -> 283.
    const int blocks = MB == 1 ? 1 : min(MB, __builtin_amdgcn_readfirstlane((mend - m0 + 32 * WM - 1) / (32 * WM)));
    static_assert(MB == 1 || DEPTH == 2, "two slots, given back by parts");
    auto request_a = [&](int slot, int a) {                    // row block a of A's next slot that it has not requested, into ring slot `slot`
#pragma unroll
        for (int i = 0; i < RA; i++) { tl_dma16(basea + slot * AS + a * (32 * WM * TL_ROW) + i * 1024u, as[a][i]); as[a][i] += BK; }
    };
    auto request_w = [&](int slot) {
#pragma unroll
        for (int i = 0; i < RW; i++) { tl_dma16(basew + slot * WS + i * 1024u, ws[i]); ws[i] += BK; }
    };
    // fragment of rows [32 blk, +32), k step ks of the slot: chunk ks + 4 h of row r (the halves of the wave take k halves of the slot; any order serves, both operands alike)
    const int sw = (4 * h) ^ ((r >> 1) & 7);
    const uint8_t* afp = ring_ + (wr * 32 + r) * TL_ROW;
    const uint8_t* wfp = ring_ + DEPTH * AS + (wc * (BN / WN) + r) * TL_ROW;
    auto multiply = [&](gv16f& c, const gu4& fa, const gu4& fb) {
        c = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(gb8, fa), __builtin_bit_cast(gb8, fb), c, 0, 0, 0);
    };
    // one block per wave, several workgroups per unit: whole slots, DEPTH deep, one barrier each; the next slot's first fragments are read during this one's last products
    auto whole_slots = [&]() {
        gu4 af[2], wf[2];
        auto request = [&](int slot) { request_a(slot, 0); request_w(slot); };
        auto read = [&](int slot, int ks) {
            af[ks & 1] = *reinterpret_cast<const gu4*>(afp + slot * AS + ((ks ^ sw) << 4));
            wf[ks & 1] = *reinterpret_cast<const gu4*>(wfp + slot * WS + ((ks ^ sw) << 4));
        };
#pragma unroll
        for (int d = 0; d < DEPTH; d++) if (d < steps) request(d);
        // a slot has landed when only the younger ones are outstanding
        if (steps >= DEPTH) tl_wait_barrier<(DEPTH - 1) * (RA + RW)>(); else tl_wait_barrier<0>();
        read(0, 0);
        int slot = 0;
        for (int s = 0; s < steps; s++) {
#pragma unroll
            for (int ks = 0; ks < 4; ks++) {
                if (ks + 1 < 4) read(slot, ks + 1);
                else if (s + 1 < steps) {
                    // the wave's last fragments of slot s are in registers: behind the barrier every wave's are
                    if (s + DEPTH - 1 < steps) tl_wait_barrier<(DEPTH - 2) * (RA + RW)>(); else tl_wait_barrier<0>();
                    const int next = slot == DEPTH - 1 ? 0 : slot + 1;
                    read(next, 0);
                    if (s + DEPTH < steps) request(slot);
                    slot = next;
                }
                __builtin_amdgcn_sched_barrier(0);
                multiply(acc[0][0], af[ks & 1], wf[ks & 1]);
                __builtin_amdgcn_sched_barrier(0);
            }
        }
    };
    // Slots by parts, for a tile of `used` row blocks.  Phase a multiplies block a's fragments with W's and reads block a + 1's; the last phase of a slot reads block 0 and W of
    // the next one instead.  Two barriers a slot, before phase 0 and before phase HB, and behind each the requests for what was read since the one before:
    //   before phase 0, slot s:    blocks HB + 1 .. of slot s + 1, block 0 and W of slot s + 2      (N1 requests of a wave)
    //   before phase HB:           blocks 1 .. HB of slot s + 2                                     (N2)
    // Each is needed behind the third barrier after it: that barrier waits until only the N1 + N2 requests made since then are outstanding (fewer at the end, where
    // slots past the last are not requested).  Fragments read for a slot past the last are whatever stands in the ring and are not multiplied.
    auto slots_by_parts = [&](auto used) {
        constexpr int MU = used(), HB = MU / 2, N2 = HB * RA, N1 = (MU - HB) * RA + RW, NT = (MU - 1 - HB) * RA;      // NT: of N1, slot s + 1's
        gu4 af[2][4], wf[4][NB];
        auto read_a = [&](int buf, int slot, int a, int ks) { af[buf][ks] = *reinterpret_cast<const gu4*>(afp + slot * AS + a * (32 * WM * TL_ROW) + ((ks ^ sw) << 4)); };
        auto read_w = [&](int slot, int ks) {
#pragma unroll
            for (int b = 0; b < NB; b++) wf[ks][b] = *reinterpret_cast<const gu4*>(wfp + slot * WS + b * (32 * TL_ROW) + ((ks ^ sw) << 4));
        };
        request_a(0, 0); request_w(0);
#pragma unroll
        for (int a = 1; a < MU; a++) request_a(0, a);
        if (steps > 1) {
            request_a(1, 0); request_w(1);
#pragma unroll
            for (int a = 1; a <= HB; a++) request_a(1, a);
            tl_wait_barrier<N1 + N2>();
        } else tl_wait_barrier<N2 + NT>();
#pragma unroll
        for (int ks = 0; ks < 4; ks++) { read_a(0, 0, 0, ks); read_w(0, ks); }
        auto step = [&](auto par_, int s) {                    // par_: s % 2, the ring slot, and with an odd number of blocks the fragment buffer of block 0
            constexpr int par = par_(), first = MU % 2 ? par : 0;
            const bool one = s + 1 < steps, two = s + 2 < steps;
            if (one) tl_wait_barrier<N1 + N2>(); else tl_wait_barrier<NT>();
            auto request = [&](int i) {                        // the first barrier's requests in three portions, between products
                if (i == 0 && one) {
#pragma unroll
                    for (int a = HB + 1; a < MU; a++) request_a(1 - par, a);
                }
                if (i == 1 && two) request_a(par, 0);
                if (i == 2 && two) request_w(par);
            };
            if (HB == 0) { request(0); request(1); request(2); }
#pragma unroll
            for (int a = 0; a < MU; a++) {
                const int buf = (a + first) & 1;
                if (a == HB) { if (two) tl_wait_barrier<N1 + N2>(); else if (one) tl_wait_barrier<N2 + NT>(); else tl_wait_barrier<0>(); }
#pragma unroll
                for (int ks = 0; ks < 4; ks++) {
#pragma unroll
                    for (int b = 0; b < NB; b++) multiply(acc[a][b], af[buf][ks], wf[ks][b]);
                    if (a + 1 < MU) read_a(buf ^ 1, par, a + 1, ks);
                    else { read_a(buf ^ 1, 1 - par, 0, ks); read_w(1 - par, ks); }
                    if (HB > 0 && a == 0) request(ks);
                    if (a == HB && ks < HB && two) request_a(par, 1 + ks);
                    __builtin_amdgcn_sched_barrier(0);
                }
            }
        };
        for (int s = 0; s < steps; s += 2) {
            step(std::integral_constant<int, 0>{}, s);
            if (s + 1 < steps) step(std::integral_constant<int, 1>{}, s + 1);
        }
    };
    using std::integral_constant;
    if constexpr (MB == 1) whole_slots();
    else if (blocks == MB) slots_by_parts(integral_constant<int, MB>{});
    else if (MB > 2 && blocks == 3) slots_by_parts(integral_constant<int, (MB > 2 ? 3 : 1)>{});
    else if (MB > 2 && blocks == 2) slots_by_parts(integral_constant<int, (MB > 2 ? 2 : 1)>{});
    else slots_by_parts(integral_constant<int, 1>{});
    if constexpr (GLU) {
        if (pairs) {
            tl_wait_barrier<0>();
            constexpr int LD = 36;                             // floats of a staged row: 16-byte pieces
            float* pg = reinterpret_cast<float*>(ring_) + wave * (2 * 32 * LD);
            float* pu = pg + 32 * LD;
            uint16_t* out = (uint16_t*)g.glu_out;
            const bool wide = g.glu_f % 8 == 0;
            const int row = lane >> 2, c8 = (lane & 3) * 8;    // a lane's eight columns of rows row and row + 16
#pragma unroll
            for (int b = 0; b < NB / 2; b++) {
                const int n = n0 + wc * (BN / WN / 2) + b * 32;
                const float bg = g.bias && n + r < N ? g.bias[g.glu_lo + n + r] : 0.0f, bu = g.bias && n + r < N ? g.bias[g.glu_lo + g.glu_f + n + r] : 0.0f;
#pragma unroll
                for (int a = 0; a < MB; a++) {
#pragma unroll
                    for (int i = 0; i < 16; i++) {
                        const int o = ((i & 3) + 8 * (i >> 2) + 4 * h) * LD + r;
                        pg[o] = acc[a][b][i] + bg; pu[o] = acc[a][b + NB / 2][i] + bu;
                    }
                    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront"); __builtin_amdgcn_wave_barrier(); __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
#pragma unroll 1
                    for (int it = 0; it < 2; it++) {
                        const int o = (row + 16 * it) * LD + c8, m = m0 + (a * WM + wr) * 32 + row + 16 * it;
                        if (m >= mend || n + c8 >= N) continue;
                        const float w = g.glu_row_w ? g.glu_row_w[m] : 1.0f;
                        float4 v0 = *reinterpret_cast<const float4*>(pg + o), v1 = *reinterpret_cast<const float4*>(pg + o + 4);
                        const float4 u0 = *reinterpret_cast<const float4*>(pu + o), u1 = *reinterpret_cast<const float4*>(pu + o + 4);
                        // x sigmoid(z) u with z = x, alpha x or, for the tanh form of gelu, 2 sqrt(2 / pi) (x + 0.044715 x^3), as 1 + tanh(z / 2) = 2 sigmoid(z).  A reciprocal
                        // refined once is as good as the division; one formula keeps the sixteen copies short (a loop over the longer ones cost 24 us of the 252)
                        const bool clamped = g.glu_kind == KR_SV_ACT_CLAMPED_SWIGLU;
                        const float alpha = clamped ? g.glu_alpha : g.glu_kind == KR_SV_ACT_GELU_TANH ? 1.5957691216057308f : 1.0f, cube = g.glu_kind == KR_SV_ACT_GELU_TANH ? 0.044715f : 0.0f;
                        const float lim = g.glu_limit, plus = clamped ? 1.0f : 0.0f;
                        auto act = [&](float x, float u) {
                            x *= w; u *= w;
                            if (clamped) { x = fminf(x, lim); u = fminf(fmaxf(u, -lim), lim); }
                            const float z = alpha * (cube != 0.0f ? x + cube * x * x * x : x);
                            const float d = 1.0f + expf(-z), q = __builtin_amdgcn_rcpf(d);
                            return x * (d < INFINITY ? __builtin_fmaf(__builtin_fmaf(-d, q, 1.0f), q, q) : 0.0f) * (u + plus);
                        };
                        v0 = make_float4(act(v0.x, u0.x), act(v0.y, u0.y), act(v0.z, u0.z), act(v0.w, u0.w));
                        v1 = make_float4(act(v1.x, u1.x), act(v1.y, u1.y), act(v1.z, u1.z), act(v1.w, u1.w));
                        const uint32_t y[8] = {kr_f32_to_bf16(v0.x), kr_f32_to_bf16(v0.y), kr_f32_to_bf16(v0.z), kr_f32_to_bf16(v0.w),
                                               kr_f32_to_bf16(v1.x), kr_f32_to_bf16(v1.y), kr_f32_to_bf16(v1.z), kr_f32_to_bf16(v1.w)};
                        uint16_t* dst = out + (size_t)m * g.glu_f + n + c8;
                        if (wide) *reinterpret_cast<gu4*>(dst) = gu4{y[0] | (y[1] << 16), y[2] | (y[3] << 16), y[4] | (y[5] << 16), y[6] | (y[7] << 16)};
                        else {
#pragma unroll
                            for (int e = 0; e < 8; e++) if (n + c8 + e < N) dst[e] = (uint16_t)y[e];
                        }
                    }
                    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront"); __builtin_amdgcn_wave_barrier(); __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
                }
            }
            return;
        }
    }
    if (!g.c_rows && !g.bias && g.silu_hi <= g.silu_lo && !g.o_gate && !g.c_storage) {
#pragma unroll
        for (int a = 0; a < MB; a++)
#pragma unroll
            for (int b = 0; b < NB; b++) {
                const int n = n0 + wc * (BN / WN) + b * 32 + r, mb = m0 + (a * WM + wr) * 32 + 4 * h;
                float* c = g.C + (size_t)mb * g.ldc + column(n);
                if (n < N) {
#pragma unroll
                    for (int i = 0; i < 16; i++) {
                        const int dm = (i & 3) + 8 * (i >> 2);
                        if (mb + dm < mend) c[(size_t)dm * g.ldc] = acc[a][b][i];
                    }
                }
            }
        return;
    }
    // bias, gates, row maps: one 32 x 32 block at a time through a wave's own piece of LDS, so that the element epilogue is a loop and not 16 MB NB copies of itself
    tl_wait_barrier<0>();
    float* blk = reinterpret_cast<float*>(ring_) + wave * (32 * 33);
#pragma unroll
    for (int a = 0; a < MB; a++)
#pragma unroll
        for (int b = 0; b < NB; b++) {
#pragma unroll
            for (int i = 0; i < 16; i++) blk[((i & 3) + 8 * (i >> 2) + 4 * h) * 33 + r] = acc[a][b][i];
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront"); __builtin_amdgcn_wave_barrier(); __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
            const int n = n0 + wc * (BN / WN) + b * 32 + r, mb = m0 + (a * WM + wr) * 32;
#pragma unroll 1
            for (int i = h; i < 32; i += 2)
                if (n < N && mb + i < mend) gm_store<true>(g, mb + i, column(n), blk[i * 33 + r]);
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront"); __builtin_amdgcn_wave_barrier(); __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        }
}

template <int BM, int BN, int WM, int WN, int DEPTH, int WPS, bool GLU>
void tl_launch(const KrSvGemm& g, hipStream_t st) {
    constexpr int LDS = DEPTH * (BM + BN) * TL_ROW;
    static_assert(LDS <= 160 * 1024, "LDS of a compute unit");
    static_assert(!GLU || (BN / WN % 64 == 0 && WM * WN * 2 * 32 * 36 * 4 <= LDS), "a wave holds both factors, and stages them");
    const int cols = GLU ? (g.N - 2 * g.glu_f + BN - 1) / BN + (g.glu_f + BN / 2 - 1) / (BN / 2) : (g.N + BN - 1) / BN;
    const dim3 grid(cols, (g.M + BM - 1) / BM + (g.seg ? g.n_groups : 0));
    if (kr_lds_optin((const void*)sv_tile_kernel<BM, BN, WM, WN, DEPTH, WPS, GLU>, LDS)) return;
    hipLaunchKernelGGL((sv_tile_kernel<BM, BN, WM, WN, DEPTH, WPS, GLU>), grid, dim3(64 * WM * WN), LDS, st, g);
}
}  // namespace

// whole slots of 16-byte chunks
bool kr_sv_gemm_tile_fits(const KrSvGemm& g, bool f32) {
    const int row = TL_ROW / (f32 ? 4 : 2), chunk = 16 / (f32 ? 4 : 2);
    return g.K % row == 0 && (!f32 || g.K < 1 << 24) && g.lda % chunk == 0 && (((uintptr_t)g.A | (uintptr_t)g.W) % 16 == 0) && g.w_stride % chunk == 0;
}

// Which tile: the time of a slot step times how often the chip has to be filled, as measured at K = 2048 - 8192 (us per step of 64 k):
// (the slots by parts take 15 - 20 % off the two larger tiles, 8 % off the small one: the choice between them is the same, within 4 % of the best of the three at 70 of 77 sizes from 40 to 1500 rows,
// 1536 to 12416 columns and 600 to 13000 expert rows)
//   256 x 256, eight waves, one workgroup per compute unit: 2.1 per round of 256 tiles, however empty the last round is
//   128 x 128, two workgroups per unit: 1.5 per 512 tiles, shares of a round cost their share (the resident workgroups slow one another), at least 0.72
//   64 x 64, three per unit: 0.4 + 0.7 per 768 tiles: few rows, where the small tile spreads the weight stream over more units
// (us, 256 / 128 / 64: 3300 x 4096 x 8192 267 / 315 / 391; 4096 x 2048 x 2048 61 / 42 / 57; 500 x 2048 x 2048 53 / 23 / 14.)  Tiles of a grouped problem: its rows spread
// evenly, half a tile more per group.
static double tl_tiles(const KrSvGemm& g, int b) {
    const double cols = (g.N + b - 1) / b;
    return cols * (g.seg ? g.n_groups * std::max(1.0, (double)g.M / g.n_groups / b + 0.5) : (double)((g.M + b - 1) / b));
}
static int tl_kind(const KrSvGemm& g) {
    const double t256 = 2.1 * std::ceil(tl_tiles(g, 256) / 256), t128 = std::max(0.72, 1.5 * tl_tiles(g, 128) / 512), t64 = 0.4 + 0.7 * tl_tiles(g, 64) / 768;
    return t256 <= t128 && t256 <= t64 ? 256 : t128 <= t64 ? 128 : 64;
}

// the two larger tiles, whose waves hold whole pairs; columns that pass other gates must lie outside the pairs
bool kr_sv_gemm_tile_glu_fits(const KrSvGemm& g) {
    return g.glu_kind != KR_SV_ACT_RELU2 && g.glu_f > 0 && g.glu_lo >= 0 && g.glu_lo + 2 * g.glu_f <= g.N && g.n_last <= 0 && !g.o_gate && !g.c_rows && !g.c_storage && (uintptr_t)g.glu_out % 16 == 0 &&
           (g.silu_hi <= g.silu_lo || g.silu_hi <= g.glu_lo || g.silu_lo >= g.glu_lo + 2 * g.glu_f) && tl_kind(g) != 64;
}

void kr_sv_gemm_tile(const KrSvGemm& g, bool f32, hipStream_t st) {
    if (f32) { kr_sv_gemm_tile_f32(g, st); return; }
    switch (tl_kind(g)) {
        case 256: if (g.glu_out) tl_launch<256, 256, 2, 4, 2, 2, true>(g, st); else tl_launch<256, 256, 2, 4, 2, 2, false>(g, st); break;
        case 128: if (g.glu_out) tl_launch<128, 128, 2, 2, 2, 2, true>(g, st); else tl_launch<128, 128, 2, 2, 2, 2, false>(g, st); break;
        default: tl_launch<64, 64, 2, 2, 3, 3, false>(g, st); break;
    }
}
