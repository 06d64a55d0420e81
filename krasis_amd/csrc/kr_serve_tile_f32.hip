// kr_serve_tile_f32.hip -- C[M, N] = A[M, K] x W[N, K]^T of an f32 store for prompt-sized problems, single matrix or one matrix per expert, every factor and sum in f32.
//
// Bound: the f32 matrix instructions (150 TFLOP/s is what a loop of them alone reaches here), with few rows per expert the weight stream.  What decides the layout:
//   * A vector instruction between two of them costs about 20 clocks (32x32x2 products with one integer add after each 29 -> 40 ns, 16x16x4 16 -> 25; bf16 products 14.9 -> 15.7), so
//     the loop has none but two pointer advances a slot: fragment addresses are fixed per lane with the slot in the instruction's offset, the weights' base is scalar.
//   * The forms with k = 1 take a fragment of four k as it lies in LDS, W's 64 columns across the lanes, and rows in any multiple of four: 16 rows of a wave are one
//     16x16x1 over four column blocks, 4, 8 or 12 rows that many 4x4x1 over sixteen.  The tile's rows are dealt to its four waves, so 35 rows cost as 48 and not as 64.
//   * Every form adds its products one k after the other (as a chain of fused multiply-adds), so all of them give the same bits.
//   * Four requests behind one another hold a wave for 16 cycles each on the unit's request path, and its products with it: one per quarter slot instead.
// Measured, us, against 64 x 64 and 128 x 128 tiles on 32x32x2 products: 64 experts, 360 / 1500 / 3000 / 9000 rows of 1536 x 2048 253 / 253 / 260 / 640 -> 160 / 171 / 262 / 617 (the last two:
// matrix instructions 70 % of the clocks, clock held at 2.0 - 2.1 GHz), of 2048 x 768 125 / 127 / 129 / 350 -> 77 / 89 / 122 / 337; 500 rows x 4160 x 2048 117 -> 99, 250 76 -> 67,
// 4000 566 -> 571 (120 TFLOP/s).  Tiles of 128 columns (half the requests): 5 % faster from 9000 expert rows on, slower wherever a single matrix has fewer than 2000.
#include <cmath>
#include <type_traits>

#include "kr_lds_optin.h"
#include "kr_serve_tile_dev.h"

namespace {
typedef float gv4f __attribute__((ext_vector_type(4)));
constexpr int TF_WAVES = 4, BN = 64, DEPTH = 3, RW = 2;        // columns, ring slots of 32 k (two: 10 - 15 % slower where weights come from memory; four: two workgroups a unit instead of three), a wave's requests for W's slot
constexpr uint32_t WS = BN * TL_ROW;

// tl_dma16 from a base that the whole wave shares, and the lane's offset in bytes
__device__ __forceinline__ void tf_dma16(uint32_t lds_dst, const void* base, uint32_t off) {
    unsigned keep;
    asm volatile("s_mov_b32 %0, m0\n\ts_mov_b32 m0, %3\n\ts_nop 2\n\tglobal_load_lds_dwordx4 %1, %2\n\ts_mov_b32 m0, %0" : "=&s"(keep) : "v"(off), "s"(base), "s"(lds_dst) : "memory");
}

// BM: rows of a tile, at most 64
__global__ void __launch_bounds__(64 * TF_WAVES, 3) sv_tile_f32_kernel(const KrSvGemm g, const int BM) {
    extern __shared__ __attribute__((aligned(1024))) uint8_t ring_[];
    int bx = blockIdx.x, by = blockIdx.y;
    // the XCDs' share of tiles: kr_serve_tile.hip
    if (g.seg || gridDim.x % 8 != 0) {
        const int gx = gridDim.x, L = by * gx + bx, band = L / (16 * gx), rem = L - band * 16 * gx, rows = min(16, (int)gridDim.y - band * 16);
        if (rows == 16) { by = band * 16 + 2 * (rem & 7) + ((rem >> 3) & 1); bx = rem >> 4; }
        else { by = band * 16 + rem % rows; bx = rem / rows; }
    }
    int group = 0, m0 = by * BM, mend = g.M;
    if (g.seg && !gm_find_tile(g.seg, g.n_groups, by, BM, group, m0, mend)) return;
    mend = min(mend, m0 + BM);
    const int n0 = bx * BN, N = gm_cols(g, group);
    if (n0 >= N) return;
    const float* A = (const float*)g.A;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int steps = g.K / 32;
    const uint32_t ringa = __builtin_amdgcn_readfirstlane(tl_lds_addr(ring_));
    auto run = [&](auto used) {
        constexpr int RB = used(), RA = (RB + 1) / 2, RQ = RA + RW;      // a wave's rows are 4 RB
        constexpr uint32_t AS = RA * 32 * TL_ROW;
        const float* as[RA]; uint32_t wo[RW];
        const uint64_t w0 = (uint64_t)(uintptr_t)((const float*)g.W + (size_t)group * g.w_stride + (size_t)n0 * g.K);
        const float* wb = (const float*)(uintptr_t)(((uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((uint32_t)(w0 >> 32)) << 32) | (uint32_t)__builtin_amdgcn_readfirstlane((uint32_t)w0));
#pragma unroll
        for (int i = 0; i < RA; i++) {
            const int row = (wave * RA + i) * 8 + (lane >> 3), ch = (lane & 7) ^ ((row >> 1) & 7), m = min(m0 + row, mend - 1);
            as[i] = A + (size_t)(g.a_rows ? g.a_rows[m] : m) * g.lda + ch * 4;
        }
#pragma unroll
        for (int i = 0; i < RW; i++) {
            const int row = (wave * RW + i) * 8 + (lane >> 3), ch = (lane & 7) ^ ((row >> 1) & 7);
            wo[i] = ((uint32_t)min(row, N - 1 - n0) * (uint32_t)g.K + ch * 4) * 4u;
        }
        const uint32_t basew = ringa + wave * RW * 1024u, basea = ringa + DEPTH * WS + wave * RA * 1024u;
        // one request of a slot; the addresses move on behind the last, in one group
        auto request = [&](int slot, int i) {
            if (i < RW) tf_dma16(basew + slot * WS + i * 1024u, wb, wo[i]);
            else tl_dma16(basea + slot * AS + (i - RW) * 1024u, as[i - RW]);
            if (i == RQ - 1) {
                wb += 32;
#pragma unroll
                for (int j = 0; j < RA; j++) as[j] += 32;
            }
        };
        const int ar = wave * 4 * RB + min(lane & 15, 4 * RB - 1), ax = (ar >> 1) & 7, wx = (lane >> 1) & 7;
        const uint8_t* ap[8]; const uint8_t* wp[8];
#pragma unroll
        for (int c = 0; c < 8; c++) { wp[c] = ring_ + lane * TL_ROW + ((c ^ wx) << 4); ap[c] = ring_ + DEPTH * WS + ar * TL_ROW + ((c ^ ax) << 4); }
        // chunk ks and chunk ks + 4 of a slot make k step ks: k = 4 ks + e and 16 + 4 ks + e in turn
        gu4 af[2][2], wf[2][2];
        auto read = [&](int slot, int ks) {
#pragma unroll
            for (int h = 0; h < 2; h++) {
                wf[ks & 1][h] = *reinterpret_cast<const gu4*>(wp[ks + 4 * h] + slot * WS);
                af[ks & 1][h] = *reinterpret_cast<const gu4*>(ap[ks + 4 * h] + slot * AS);
            }
        };
        gv16f acc;
        gv4f quad[4];
#pragma unroll
        for (int i = 0; i < 16; i++) { acc[i] = 0.0f; quad[i / 4][i % 4] = 0.0f; }
        auto multiply = [&](int buf, int e0) {
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int e = e0; e < e0 + 2; e++)
#pragma unroll
                for (int h = 0; h < 2; h++) {
                    const float a = __uint_as_float(af[buf][h][e]), w = __uint_as_float(wf[buf][h][e]);
                    if constexpr (RB == 4) acc = __builtin_amdgcn_mfma_f32_16x16x1f32(a, w, acc, 2, 0, 0);
                    else {
                        quad[0] = __builtin_amdgcn_mfma_f32_4x4x1f32(a, w, quad[0], 4, 0, 0);
                        if constexpr (RB > 1) quad[1] = __builtin_amdgcn_mfma_f32_4x4x1f32(a, w, quad[1], 4, 1, 0);
                        if constexpr (RB > 2) quad[2] = __builtin_amdgcn_mfma_f32_4x4x1f32(a, w, quad[2], 4, 2, 0);
                    }
                }
            __builtin_amdgcn_sched_barrier(0);
        };
        // Slot s + 1 has landed when only the slots behind it are outstanding.  A slot is free behind the barrier of its last quarter; it is requested again in that one and the next three.
#pragma unroll
        for (int d = 0; d < DEPTH; d++)
            if (d < steps) {
#pragma unroll
                for (int i = 0; i < RQ; i++) request(d, i);
            }
        if (steps >= DEPTH) tl_wait_barrier<(DEPTH - 1) * RQ>(); else tl_wait_barrier<0>();
        read(0, 0);
        auto step = [&](auto slot_, int s) {
            constexpr int slot = slot_(), next = (slot + 1) % DEPTH, prev = (slot + DEPTH - 1) % DEPTH;
            const bool ask = s > 0 && s - 1 + DEPTH < steps;
#pragma unroll
            for (int ks = 0; ks < 3; ks++) {
                read(slot, ks + 1);
                multiply(ks & 1, 0);
                if (ask && ks + 1 < RQ) request(prev, ks + 1);
                multiply(ks & 1, 2);
            }
            if (s + 1 < steps) { if (s + DEPTH - 1 < steps) tl_wait_barrier<(DEPTH - 2) * RQ>(); else tl_wait_barrier<0>(); }
            multiply(1, 0);
            if (s + 1 < steps) read(next, 0);
            if (s + DEPTH < steps) request(slot, 0);
            multiply(1, 2);
        };
        for (int s = 0; s < steps; s += DEPTH) {
            step(std::integral_constant<int, 0>{}, s);
            if (s + 1 < steps) step(std::integral_constant<int, 1>{}, s + 1);
            if (s + 2 < steps) step(std::integral_constant<int, 2>{}, s + 2);
        }
        // element i of a lane: 16x16x1 holds 16 rows x 16 columns four times, 4x4x1 a lane's column and four rows
        auto row = [&](int i) { return m0 + wave * 4 * RB + (RB == 4 ? 4 * (lane >> 4) + (i & 3) : i); };
        auto col = [&](int i) { return n0 + (RB == 4 ? (i & ~3) * 4 + (lane & 15) : lane); };
        auto value = [&](int i) { return RB == 4 ? acc[i] : quad[i / 4][i % 4]; };
        if (!g.c_rows && !g.bias && g.silu_hi <= g.silu_lo && !g.o_gate) {
#pragma unroll
            for (int i = 0; i < 4 * RB; i++)
                if (row(i) < mend && col(i) < N) g.C[(size_t)row(i) * g.ldc + col(i)] = value(i);
            return;
        }
        // bias, gates, row maps: through a lane's own words of LDS, so that the element epilogue is a loop and not copies of itself
        tl_wait_barrier<0>();
        float* blk = reinterpret_cast<float*>(ring_) + threadIdx.x;
#pragma unroll
        for (int i = 0; i < 4 * RB; i++) blk[i * 64 * TF_WAVES] = value(i);
#pragma unroll 1
        for (int i = 0; i < 4 * RB; i++)
            if (row(i) < mend && col(i) < N) gm_store<false>(g, row(i), col(i), blk[i * 64 * TF_WAVES]);
    };
    using std::integral_constant;
    switch (__builtin_amdgcn_readfirstlane((mend - m0 + 15) / 16)) {
        case 1: run(integral_constant<int, 1>{}); break;
        case 2: run(integral_constant<int, 2>{}); break;
        case 3: run(integral_constant<int, 3>{}); break;
        default: run(integral_constant<int, 4>{}); break;
    }
}
}  // namespace

// Rows of a tile, by the time of the fullest unit: rounds of 256 tiles times a tile's row blocks, and 15 % for a smaller tile, whose weights are read more often.  Experts
// take 64: a tile costs the blocks it has.  (us, 64 / 48 / 32: 500 rows x 4160 x 2048 113 / 99 / 111, x 2048 47 / 67 / 52; 250 x 4160 74 / 67 / 66, x 2048 43 / 46 / 34; 1500 x 2048 121 / 140 / 132.)
static int tf_rows(const KrSvGemm& g) {
    int best = 64; double least = 0.0;
    for (int bm = 64; bm >= 32 && !g.seg; bm -= 16) {
        const double t = std::ceil((double)((g.N + BN - 1) / BN) * ((g.M + bm - 1) / bm) / 256) * bm * (bm == 64 ? 1.0 : 1.15);
        if (bm == 64 || t < least) { least = t; best = bm; }
    }
    return best;
}

// K whole slots, below 2^24: a lane's offset in its tile of W is 32 bits (kr_sv_gemm_tile_fits)
void kr_sv_gemm_tile_f32(const KrSvGemm& g, hipStream_t st) {
    const int bm = tf_rows(g), lds = DEPTH * ((bm + 31) / 32 * 32 + BN) * TL_ROW;
    const dim3 grid((g.N + BN - 1) / BN, (g.M + bm - 1) / bm + (g.seg ? g.n_groups : 0));
    if (kr_lds_optin((const void*)sv_tile_f32_kernel, lds)) return;
    hipLaunchKernelGGL(sv_tile_f32_kernel, grid, dim3(64 * TF_WAVES), lds, st, g, bm);
}
