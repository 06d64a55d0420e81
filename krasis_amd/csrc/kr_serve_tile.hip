// kr_serve_tile.hip -- C[M, N] = A[M, K] x W[N, K]^T for prompt-sized problems of a bf16 store, single matrix or one matrix per expert, on v_mfma_f32_32x32x16_bf16.
//
// Bound: the matrix cores (about 1350 TFLOP/s is what a large library product reaches here; nominal 2500).  Both operands travel from memory to LDS by
// global_load_lds_dwordx4 into a ring of slots of 64 k (no staging registers; whole cache lines), ONE barrier per slot, the next slot requested right behind it, fragments
// of a k step read while the step before is multiplied.  What the large tile buys: 256 x 256 by eight waves of 128 x 64 reads 48 KB of fragments per 64 matrix
// instructions and SIMD and 64 KB of operands per slot; 128 x 128 by four waves of 64 x 64 needs a third more of the first and twice the second for the same products,
// and neither the LDS nor the L2 rate hides behind the matrix cores then (requests and reads without products 206 us, products without requests 197 us, both 315 us at
// 3300 x 4096 x 8192).  LDS-DMA writes lane-linear (lane i at base + 16 i), so bank conflicts are avoided on the SOURCE side: the 16-byte chunk c of row r sits at
// position c ^ (r / 2 % 8) of its 128-byte row and the fragment reads apply the same map (without it 1.6 - 2.1 x slower).
// Measured, us, register-staged 128 x 128 tile before -> now: 3300 x 4096 x 8192 425 -> 238 (931 TFLOP/s), 3300 x 12544 x 4096 596 -> 376, 4096 x 4224 x 2048 144 -> 104,
// 64 experts 24576 x 1536 x 2048 372 -> 248 and x 2048 x 768 217 -> 149, 500 x 2048 x 2048 36.8 -> 14.1, 100 x 4224 x 2048 36.9 -> 13.2.
#include <algorithm>
#include <cmath>

#include "kr_serve_gemm_dev.h"

namespace {
constexpr int TL_BK = 64;                                      // k of a slot: 128-byte rows, whole cache lines (32 k would fetch every line twice)

__device__ __forceinline__ uint32_t tl_lds_addr(const void* p) { return (uint32_t)(uintptr_t)(const __attribute__((address_space(3))) char*)p; }
// 64 lanes x 16 bytes from the lane's own address to lds_dst (wave-uniform) + 16 lane.  M0 is the compiler's register: saved and restored inside.  The compiler
// does not count this request; the waits below do.
__device__ __forceinline__ void tl_dma16(uint32_t lds_dst, const uint16_t* src) {
    unsigned keep;
    asm volatile("s_mov_b32 %0, m0\n\ts_mov_b32 m0, %2\n\ts_nop 2\n\tglobal_load_lds_dwordx4 %1, off\n\ts_mov_b32 m0, %0" : "=&s"(keep) : "v"(src), "s"(lds_dst) : "memory");
}
// at most N of this wave's requests are outstanding and its LDS reads have returned, then the workgroup barrier
template <int N> __device__ __forceinline__ void tl_wait_barrier() { asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" :: "n"(N) : "memory"); }

template <int BM, int BN, int WM, int WN, int DEPTH, int WPS>  // WM x WN waves; WPS: waves per SIMD the register budget is for
__global__ void __launch_bounds__(64 * WM * WN, WPS) sv_tile_kernel(const KrSvGemm g) {
    constexpr int MB = BM / (32 * WM), NB = BN / (32 * WN);    // 32 x 32 blocks of a wave
    constexpr int RA = BM / 8, RW = (BM + BN) / (8 * WM * WN); // requests of 8 rows per slot: A's; per wave
    constexpr int SLOT = (BM + BN) * TL_BK;                    // elements
    extern __shared__ __attribute__((aligned(1024))) uint16_t ring[];
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
    const int n0 = bx * BN, N = gm_cols(g, group);
    if (n0 >= N) return;
    const uint16_t* A = (const uint16_t*)g.A;
    const uint16_t* W = (const uint16_t*)g.W + (size_t)group * g.w_stride;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), r = lane & 31, h = lane >> 5, wr = wave / WN, wc = wave % WN;
    const uint16_t* src[RW];
#pragma unroll
    for (int i = 0; i < RW; i++) {
        const int q = wave * RW + i;                           // request: RA of A's rows, then W's
        const int row = (q < RA ? q : q - RA) * 8 + (lane >> 3), ch = (lane & 7) ^ ((row >> 1) & 7);
        if (q < RA) { const int m = min(m0 + row, mend - 1); src[i] = A + (size_t)(g.a_rows ? g.a_rows[m] : m) * g.lda + ch * 8; }
        else src[i] = W + (size_t)min(n0 + row, N - 1) * g.K + ch * 8;
    }
    const uint32_t base = __builtin_amdgcn_readfirstlane(tl_lds_addr(ring)) + (uint32_t)(wave * RW) * 1024u;
    gv16f acc[MB][NB];
#pragma unroll
    for (int a = 0; a < MB; a++)
#pragma unroll
        for (int b = 0; b < NB; b++)
#pragma unroll
            for (int i = 0; i < 16; i++) acc[a][b][i] = 0.0f;
    const int steps = g.K / TL_BK;
    auto request = [&](int slot) {
#pragma unroll
        for (int i = 0; i < RW; i++) { tl_dma16(base + (uint32_t)slot * (SLOT * 2) + i * 1024u, src[i]); src[i] += TL_BK; }
    };
#pragma unroll
    for (int d = 0; d < DEPTH - 1; d++) if (d < steps) request(d);
    // fragment of rows [32 blk, +32), k step ks of the slot: chunk ks + 4 h of row r
    const int sw = (r >> 1) & 7;
    const uint16_t* af0 = ring + (wr * (BM / WM) + r) * TL_BK;
    const uint16_t* bf0 = ring + (BM + wc * (BN / WN) + r) * TL_BK;
    int slot = 0;
    for (int s = 0; s < steps; s++) {
        // slot s has landed when only the DEPTH - 2 younger ones are outstanding (none at the end)
        if (DEPTH == 2 || s + 1 >= steps) tl_wait_barrier<0>(); else tl_wait_barrier<(DEPTH - 2) * RW>();
        if (s + DEPTH - 1 < steps) request(slot == 0 ? DEPTH - 1 : slot - 1);      // the slot read in the previous step: every wave is past it
        const uint16_t* ab = af0 + slot * SLOT;
        const uint16_t* bb = bf0 + slot * SLOT;
        gb8 af[2][MB], bf[2][NB];                              // fragments of two k steps: one is read while the other is multiplied
        auto read = [&](int ks) {
            const int ch = ((ks + 4 * h) ^ sw) * 8;            // the halves of the wave take k halves of the slot (any order serves, both operands alike)
#pragma unroll
            for (int a = 0; a < MB; a++) af[ks & 1][a] = __builtin_bit_cast(gb8, *reinterpret_cast<const gu4*>(ab + a * 32 * TL_BK + ch));
#pragma unroll
            for (int b = 0; b < NB; b++) bf[ks & 1][b] = __builtin_bit_cast(gb8, *reinterpret_cast<const gu4*>(bb + b * 32 * TL_BK + ch));
        };
        read(0);
#pragma unroll
        for (int ks = 0; ks < TL_BK / 16; ks++) {
            if (ks + 1 < TL_BK / 16) read(ks + 1);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int a = 0; a < MB; a++)
#pragma unroll
                for (int b = 0; b < NB; b++) acc[a][b] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(af[ks & 1][a], bf[ks & 1][b], acc[a][b], 0, 0, 0);
            __builtin_amdgcn_sched_barrier(0);
        }
        slot = slot == DEPTH - 1 ? 0 : slot + 1;
    }
    if (!g.c_rows && !g.bias && g.silu_hi <= g.silu_lo && !g.o_gate && !g.c_storage) {
#pragma unroll
        for (int a = 0; a < MB; a++)
#pragma unroll
            for (int b = 0; b < NB; b++) {
                const int n = n0 + wc * (BN / WN) + b * 32 + r, mb = m0 + wr * (BM / WM) + a * 32 + 4 * h;
                float* c = g.C + (size_t)mb * g.ldc + n;
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
    float* blk = reinterpret_cast<float*>(ring) + wave * (32 * 33);
#pragma unroll
    for (int a = 0; a < MB; a++)
#pragma unroll
        for (int b = 0; b < NB; b++) {
#pragma unroll
            for (int i = 0; i < 16; i++) blk[((i & 3) + 8 * (i >> 2) + 4 * h) * 33 + r] = acc[a][b][i];
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront"); __builtin_amdgcn_wave_barrier(); __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
            const int n = n0 + wc * (BN / WN) + b * 32 + r, mb = m0 + wr * (BM / WM) + a * 32;
#pragma unroll 1
            for (int i = h; i < 32; i += 2)
                if (n < N && mb + i < mend) gm_store<true>(g, mb + i, n, blk[i * 33 + r]);
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront"); __builtin_amdgcn_wave_barrier(); __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        }
}

template <int BM, int BN, int WM, int WN, int DEPTH, int WPS>
void tl_launch(const KrSvGemm& g, hipStream_t st) {
    constexpr int LDS = DEPTH * (BM + BN) * TL_BK * 2;
    static_assert(LDS <= 160 * 1024, "LDS of a compute unit");
    const dim3 grid((g.N + BN - 1) / BN, (g.M + BM - 1) / BM + (g.seg ? g.n_groups : 0));
    (void)hipFuncSetAttribute((const void*)sv_tile_kernel<BM, BN, WM, WN, DEPTH, WPS>, hipFuncAttributeMaxDynamicSharedMemorySize, LDS);
    hipLaunchKernelGGL((sv_tile_kernel<BM, BN, WM, WN, DEPTH, WPS>), grid, dim3(64 * WM * WN), LDS, st, g);
}
}  // namespace

// whole slots of 16-byte chunks
bool kr_sv_gemm_tile_fits(const KrSvGemm& g) {
    return g.K % TL_BK == 0 && g.lda % 8 == 0 && (((uintptr_t)g.A | (uintptr_t)g.W) % 16 == 0) && g.w_stride % 8 == 0;
}

// Which tile: the time of a slot step times how often the chip has to be filled, as measured at K = 2048 - 8192 (us per step of 64 k):
//   256 x 256, eight waves, one workgroup per compute unit: 2.1 per round of 256 tiles, however empty the last round is
//   128 x 128, two workgroups per unit: 1.5 per 512 tiles, shares of a round cost their share (the resident workgroups slow one another), at least 0.72
//   64 x 64, three per unit: 0.4 + 0.7 per 768 tiles: few rows, where the small tile spreads the weight stream over more units
// (us, 256 / 128 / 64: 3300 x 4096 x 8192 267 / 315 / 391; 4096 x 2048 x 2048 61 / 42 / 57; 500 x 2048 x 2048 53 / 23 / 14.)  Tiles of a grouped problem: its rows spread
// evenly, half a tile more per group.
static int tl_kind(const KrSvGemm& g) {
    auto tiles = [&](int b) {
        const double cols = (g.N + b - 1) / b;
        return cols * (g.seg ? g.n_groups * std::max(1.0, (double)g.M / g.n_groups / b + 0.5) : (double)((g.M + b - 1) / b));
    };
    const double t256 = 2.1 * std::ceil(tiles(256) / 256), t128 = std::max(0.72, 1.5 * tiles(128) / 512), t64 = 0.4 + 0.7 * tiles(64) / 768;
    return t256 <= t128 && t256 <= t64 ? 256 : t128 <= t64 ? 128 : 64;
}

void kr_sv_gemm_tile(const KrSvGemm& g, hipStream_t st) {
    switch (tl_kind(g)) {
        case 256: tl_launch<256, 256, 2, 4, 2, 2>(g, st); break;
        case 128: tl_launch<128, 128, 2, 2, 2, 2>(g, st); break;
        default: tl_launch<64, 64, 2, 2, 3, 3>(g, st); break;
    }
}
