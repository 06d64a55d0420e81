// kr_prefill_w.hip -- the tolerance GEMM of the prompt pass (KR_GEMM_FAST), INT4 weights, for problems that fill the chip: f16 rows x weights de-quantized in registers on
// v_mfma_f32_32x32x16_f16, f32 accumulation over the whole k range.  Same products and the same order of sums per output as kr_pfh_gemm_kernel (kr_prefill_h.hip): the same bits.
//
// Bound: the matrix cores and, beside them, the vector port, which turns every weight into f16 once per tile: 12 instructions per 32 columns and 16 k, 24 for a wave's two column blocks, whatever the tile's rows.  So a
// wave multiplies them by three row blocks (4 - 5 vector instructions per matrix instruction; two blocks: 7.8, with the rows' way through registers), and a tile takes the
// 80 rows that an expert of 512 has of 4096 tokens as three blocks of 32 where two tiles of 64 were four blocks and formed the weights twice.
// What travels, and how:
//   * the wave's own 64 columns: whole 128-byte lines of the resident layout by LDS-DMA into 8 KB that no other wave reads, from there to registers at the start of a stage (256 k);
//     the next stage's take their place at once, a stage of time ahead, and need no barrier;
//   * the rows, 64 k (a line) at a time: a ring of three slots that all waves share, one barrier a line, requested two lines ahead, fragments one step ahead;
//   * nothing in the loop is a vector load that the compiler counts, so every wait is a count of requests and none drains the ring.
// 74 KB of LDS and 216 registers: two workgroups a compute unit, one's start and store under the other's products.  The store goes through LDS for 16 bytes a lane.
// Measured, us, kr_pfh_gemm_kernel -> here (one MI355X, under lasting load): 512 experts, top 10, 4096 tokens 2048 -> 2 x 512 with the activation 431 -> 311, 512 -> 2048 242 -> 183; 8192 tokens 645 -> 523,
// 384 -> 338; 64 experts, top 6, 3000 tokens 2048 -> 2 x 1408 375 -> 307, 1408 -> 2048 192 -> 147; dense, 4096 rows, 2048 -> 12288 308 -> 256 (800 TFLOP/s), 4096 -> 2048 103 -> 91.
// Clocks of a compute unit at the first: 586 k -> 412 k, of them matrix instructions 255 k -> 196 k.  Tolerance prompts, ms: 8192 tokens 11.68 -> 10.4, 4096 6.07 -> 5.66, 1500 3.11 -> 2.89, 700 2.47 -> 2.11.
#include <hip/hip_runtime.h>
#include <stdint.h>
#include <type_traits>

#include "kr_lds_optin.h"
#include "kr_pfh_dev.h"
#include "kr_prefill.h"

namespace {
constexpr int BM = KR_PFW_ROWS, BN = 256, NB = BM / 32, NC = 2, DA = 3;      // rows and columns of a tile, row blocks, column blocks of a wave, slots of the row ring
constexpr int A_SLOT = BM * 128, B_WAVE = 8192, S_SLOT = 2048;               // bytes: 64 k of the rows; a wave's columns for 256 k; the group scales of a stage
constexpr int OFF_A = 0, OFF_B = OFF_A + DA * A_SLOT, OFF_S = OFF_B + 4 * B_WAVE, OFF_RM = OFF_S + 2 * S_SLOT, OFF_RD = OFF_RM + BM * 4, OFF_RS = OFF_RD + BM * 4, LDS_BYTES = OFF_RS + BM * 4;
static_assert(2 * LDS_BYTES <= 160 * 1024, "two workgroups to a compute unit");

__device__ __forceinline__ uint32_t pw_lds_addr(const void* p) { return (uint32_t)(uintptr_t)(const __attribute__((address_space(3))) char*)p; }
__device__ __forceinline__ const void* pw_uniform(const void* p) {           // the operands below must sit in scalar registers: no-ops when the compiler already knows
    const uint64_t v = (uint64_t)(uintptr_t)p;
    const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)v), hi = __builtin_amdgcn_readfirstlane((uint32_t)(v >> 32));
    return (const void*)(uintptr_t)(((uint64_t)hi << 32) | lo);
}
// 64 lanes x 16 (4) bytes from base + the lane's offset to dst + 16 (4) lane.  M0 is the compiler's register: saved and restored inside.  The compiler does not count these
// requests; the waits below do, and the loop holds no other vector load.
__device__ __forceinline__ void pw_dma16(uint32_t dst, uint32_t off, const void* base) {
    unsigned keep;
    dst = __builtin_amdgcn_readfirstlane(dst); base = pw_uniform(base);
    asm volatile("s_mov_b32 %0, m0\n\ts_mov_b32 m0, %2\n\ts_nop 2\n\tglobal_load_lds_dwordx4 %1, %3\n\ts_mov_b32 m0, %0" : "=&s"(keep) : "v"(off), "s"(dst), "s"(base) : "memory");
}
__device__ __forceinline__ void pw_dma4(uint32_t dst, uint32_t off, const void* base) {
    unsigned keep;
    dst = __builtin_amdgcn_readfirstlane(dst); base = pw_uniform(base);
    asm volatile("s_mov_b32 %0, m0\n\ts_mov_b32 m0, %2\n\ts_nop 2\n\tglobal_load_lds_dword %1, %3\n\ts_mov_b32 m0, %0" : "=&s"(keep) : "v"(off), "s"(dst), "s"(base) : "memory");
}
// at most N of this wave's requests are outstanding and its LDS reads have returned, then the workgroup barrier
template <int N> __device__ __forceinline__ void pw_wait_barrier() { asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" :: "n"(N) : "memory"); }

// A stage is 256 k (a pair of groups), a quarter of it the 64 k that a 128-byte line of a row holds.
__global__ void __launch_bounds__(256, 2) kr_pfw_gemm_kernel(const KrPfGemmHArgs a) {
    extern __shared__ __attribute__((aligned(1024))) char smem[];
    float* rmul = reinterpret_cast<float*>(smem + OFF_RM);
    int* row_dst = reinterpret_cast<int*>(smem + OFF_RD);
    uint32_t* row_src = reinterpret_cast<uint32_t*>(smem + OFF_RS);          // byte offset of every tile row in the row image
    const bool actf = a.act_fused != 0;                                      // N = 2 I, I % 128 == 0 (the launcher checks): a tile = 128 gate columns and the 128 up columns that belong to them
    const int ncb0 = (a.m.N + BN - 1) / BN, ncb1 = a.n_extra > 0 ? (a.mx[0].N + BN - 1) / BN : 0, ncb2 = a.n_extra > 1 ? (a.mx[1].N + BN - 1) / BN : 0;
    const int ncb = ncb0 + ncb1 + ncb2, xcd = blockIdx.x & 7, slot0 = blockIdx.x >> 3;
    int mt, cb;
    if (a.single_expert) {       // dense: every XCD takes an equal part of the tiles in an order that walks panels of eight column blocks row tile by row tile (their weights stay in its L2)
        const int nrt = (a.total_rows + BM - 1) / BM, tiles = nrt * ncb, per = (tiles + 7) / 8, i = xcd * per + slot0;
        if (slot0 >= per || i >= tiles) return;
        const int panel = i / (8 * nrt), w = min(8, ncb - 8 * panel), j = i - panel * 8 * nrt;
        mt = j / w; cb = panel * 8 + j - mt * w;
    } else {
        const int per = ncb * a.run, grp = slot0 / per, local = slot0 - grp * per;
        mt = (grp * 8 + xcd) * a.run + local / ncb; cb = local % ncb;
    }
    int expert, row0, rows;
    if (a.single_expert) { expert = 0; row0 = mt * BM; rows = min(BM, a.total_rows - row0); }
    else { if (mt >= a.n_tiles[0]) return; expert = a.tile_expert[mt]; row0 = a.tile_row0[mt]; rows = a.tile_rows[mt]; }
    KrMatDev m = a.m; float* out_p = a.out; int out_ld = a.out_ld;
    if (cb >= ncb0 + ncb1) { cb -= ncb0 + ncb1; m = a.mx[1]; out_p = a.outx[1]; out_ld = a.out_ldx[1]; }
    else if (cb >= ncb0) { cb -= ncb0; m = a.mx[0]; out_p = a.outx[0]; out_ld = a.out_ldx[0]; }
    const int n0 = cb * BN, half_n = m.N >> 1, n0h = cb * 128, K = m.ng * 128, nst = m.ngp;
    const char* wq = reinterpret_cast<const char*>(m.q) + (size_t)expert * m.q_stride;
    const char* wsc = reinterpret_cast<const char*>(m.s) + (size_t)expert * m.s_stride;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), n31 = lane & 31, khalf = lane >> 5;

    // a wave's 2 x 32 columns: consecutive, or (fused activation) 32 gates and the up columns that belong to them.  Column tiles past the last one read the last again (never stored).
    const int last_tile = (m.N - 1) >> 3;
    int col[NC];
    uint32_t soff[NC], brec[NC][4];                                          // the lane's scale words; a wave's records of eight columns
#pragma unroll
    for (int c = 0; c < NC; c++) {
        const int first = actf ? c * half_n + n0h + wave * 32 : n0 + wave * 64 + c * 32;
        col[c] = first + n31;
        const int cc = min(col[c], m.N - 1);
        soff[c] = (uint32_t)((cc >> 3) * nst * 8 + (cc & 7)) * 4u;
#pragma unroll
        for (int q = 0; q < 4; q++) brec[c][q] = (uint32_t)__builtin_amdgcn_readfirstlane(min((first >> 3) + q, last_tile) * nst * 1024);
    }
    const uint32_t lds0 = __builtin_amdgcn_readfirstlane(pw_lds_addr(smem));
    // Record q of a column block lands at q * 1024: lane i at column i >> 3 of it, position i & 7, where chunk (i & 7) ^ (column / 2 % 8) stands (the reads below apply the same map)
    const uint32_t bvo0 = (uint32_t)((lane >> 3) * 128 + ((lane & 7) ^ (lane >> 4)) * 16), bvo1 = bvo0 ^ 64u;
    auto request_b = [&](int st, int c) {
#pragma unroll
        for (int q = 0; q < 4; q++) pw_dma16(lds0 + OFF_B + wave * B_WAVE + c * 4096 + q * 1024, q & 1 ? bvo1 : bvo0, wq + (size_t)st * 1024 + brec[c][q]);
    };
    auto request_s = [&](int st) {
#pragma unroll
        for (int c = 0; c < NC; c++) pw_dma4(lds0 + OFF_S + (st & 1) * S_SLOT + wave * 512 + c * 256, soff[c], wsc + (size_t)st * 32);
    };
    // the first weights before the chain of dependent loads that leads to the rows; the waves that walk it, whose counter works in order, after it
    if (wave >= (BM + 63) / 64) { request_b(0, 0); request_b(0, 1); request_s(0); }
    if (tid < BM) {
        int src = -1;
        if (tid < rows) {
            if (a.single_expert) src = row0 + tid;
            else { const int pair = a.row_pair[row0 + tid]; src = a.gather_tokens ? pair / a.topk : row0 + tid; }
        }
        row_src[tid] = (uint32_t)max(src, 0) * (uint32_t)(K * 2);            // rows past `rows`: row 0
        row_dst[tid] = (a.scatter_rows && !a.single_expert && tid < rows) ? a.row_pair[row0 + tid] : row0 + tid;
        rmul[tid] = a.out_bf16 == 2 || src < 0 ? 1.0f : a.a_mul[src];        // f16 rows carry the raw accumulators: the combine pass applies the row multiplier
    }
    __syncthreads();
    if (wave < (BM + 63) / 64) { request_b(0, 0); request_b(0, 1); request_s(0); }
    // request of row block b: lane i row 8 wave + (i >> 3) of the block, position i & 7, which holds chunk (i & 7) ^ (row / 2 % 8) of the row's line
    uint32_t avo[NB];
#pragma unroll
    for (int b = 0; b < NB; b++) avo[b] = row_src[b * 32 + wave * 8 + (lane >> 3)] + (uint32_t)(((lane & 7) ^ (4 * (wave & 1) + (lane >> 4))) * 16);
    const char* abase = reinterpret_cast<const char*>(a.a);
    v16f acc[NB][NC];
#pragma unroll
    for (int b = 0; b < NB; b++)
#pragma unroll
        for (int c = 0; c < NC; c++)
#pragma unroll
            for (int r = 0; r < 16; r++) acc[b][c][r] = 0.0f;
    uint32_t M0 = 0x000F000Fu, M1 = 0x00F000F0u, MH = 0x03C003C0u, Kc = 0x64006400u;      // de-quantization masks, kept in registers (see pfh_dq4)
    asm volatile("" : "+v"(M0), "+v"(M1), "+v"(MH), "+v"(Kc));
    const int nl = 4 * nst - ((m.ng & 1) ? 2 : 0);                           // lines of 64 k
    const int sw = (n31 >> 1) & 7;

    auto main_loop = [&](auto nsa) {                                         // nsa: row blocks of this tile
        constexpr int NS = nsa();
        auto request_a = [&](int L, int slot) {
#pragma unroll
            for (int b = 0; b < NS; b++) pw_dma16(lds0 + OFF_A + slot * A_SLOT + b * 4096 + wave * 1024, avo[b], abase + (size_t)L * 128);
        };
        v8h af[2][NS], bf[2][NC];
        u32x4 raw[4][NC];                                                    // a stage of the wave's weights: record j holds words h of both groups
        v2h sq[2][NC], cq[2][NC];
        auto read_a = [&](int slot, int i) {                                 // fragments of k step i of a line: chunk 2 (i & 2) + 2 khalf + (i & 1)
            const char* p = smem + OFF_A + slot * A_SLOT + n31 * 128 + (((2 * (i & 2) + 2 * khalf + (i & 1)) ^ sw) << 4);
#pragma unroll
            for (int b = 0; b < NS; b++) af[i & 1][b] = *reinterpret_cast<const v8h*>(p + b * 4096);
        };
        auto read_b = [&]() {
            const char* p = smem + OFF_B + wave * B_WAVE + n31 * 128;
#pragma unroll
            for (int j = 0; j < 4; j++)
#pragma unroll
                for (int c = 0; c < NC; c++) raw[j][c] = *reinterpret_cast<const u32x4*>(p + c * 4096 + (((2 * j + khalf) ^ sw) << 4));
        };
        auto read_s = [&](int st) {
#pragma unroll
            for (int c = 0; c < NC; c++) {
                const uint32_t w = *reinterpret_cast<const uint32_t*>(smem + OFF_S + (st & 1) * S_SLOT + wave * 512 + c * 256 + lane * 4);
#pragma unroll
                for (int hh = 0; hh < 2; hh++) {
                    const _Float16 s1 = (_Float16)(__uint_as_float((hh ? w >> 16 : w & 0xFFFFu) << 16) * 0.25f), c1 = (_Float16)(-1536.0f * (float)s1);
                    sq[hh][c] = v2h{s1, s1}; cq[hh][c] = v2h{c1, c1};
                }
            }
        };
        // k step i of line x of a stage: group x >> 1, record 2 (x & 1) + (i >> 1), word i & 1
        auto quant = [&](int x, int i, int c) {
            const int hh = x >> 1;
            bf[i & 1][c] = pfh_dq4(raw[2 * (x & 1) + (i >> 1)][c][2 * hh + (i & 1)], sq[hh][c], cq[hh][c], M0, M1, MH, Kc);
        };
        request_a(0, 0); request_a(1, 1);
        if (nl > 2) { request_a(2, 2); pw_wait_barrier<2 * NS>(); } else pw_wait_barrier<NS>();
        read_b(); read_s(0); read_a(0, 0);
#pragma unroll
        for (int c = 0; c < NC; c++) quant(0, 0, c);
        int slot = 0;
        for (int st = 0; st < nst; st++) {
            const bool more = st + 1 < nst;
#pragma unroll
            for (int x = 0; x < 4; x++) {
                const int L = 4 * st + x, next = slot == DA - 1 ? 0 : slot + 1;
                if (x == 2 && L >= nl) break;                                // an odd number of groups
                const bool end = x == 3 ? !more : x == 1 ? L + 1 >= nl : false;
#pragma unroll
                for (int i = 0; i < 4; i++) {
                    if (i < 3) read_a(slot, i + 1);
                    else if (!end) {
                        // Every wave's last fragments of line L are in registers behind the barrier, and line L + 1 has landed (and the next stage's weights, after the last line).
                        // Requests that may be outstanding, youngest first: line L + 2 or what followed line L + 1; in the first two lines of a stage the next stage's weights too.
                        if (x < 2) { if (more) pw_wait_barrier<NS + 10>(); else if (L + 2 < nl) pw_wait_barrier<NS>(); else pw_wait_barrier<0>(); }
                        else if (more) pw_wait_barrier<NS>(); else pw_wait_barrier<0>();
                        read_a(next, 0);
                        if (x == 3) { read_b(); read_s(st + 1); }
                        if (L + 3 < nl) request_a(L + 3, slot);
                    }
                    if (x == 0 && more && i > 0) {                           // the stage's weights stand in registers: the next stage's take their place
                        if (i == 1) { asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory"); request_b(st + 1, 0); }
                        if (i == 2) { request_b(st + 1, 1); request_s(st + 1); }
                    }
                    const int xn = i < 3 ? x : (x + 1) & 3, in = (i + 1) & 3;
#pragma unroll
                    for (int c = 0; c < NC; c++)
#pragma unroll
                        for (int b = 0; b < NS; b++) acc[b][c] = __builtin_amdgcn_mfma_f32_32x32x16_f16(af[i & 1][b], bf[i & 1][c], acc[b][c], 0, 0, 0);
#pragma unroll
                    for (int c = 0; c < NC; c++) quant(xn, in, c);
                    // fragment reads, then a matrix instruction and its share of the next fragments' vector instructions in turn
                    __builtin_amdgcn_sched_group_barrier(0x100, NS, 0);
#pragma unroll
                    for (int q = 0; q < NC * NS; q++) {
                        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                        __builtin_amdgcn_sched_group_barrier(0x002, 24 / (NC * NS) + 1, 0);
                    }
                    __builtin_amdgcn_sched_barrier(0);
                }
                slot = next;
            }
        }
    };
    const int nsb = (rows + 31) / 32;
    if (nsb == NB) main_loop(std::integral_constant<int, NB>{});
    else if (nsb == 2) main_loop(std::integral_constant<int, 2>{});
    else main_loop(std::integral_constant<int, 1>{});
    // Whole and aligned columns: a wave takes its sums through LDS, 32 rows at a time, and stores 16 bytes of a row per lane.
    const int oc = actf ? a.m.N >> 1 : m.N, c0 = actf ? n0h + wave * 32 : n0 + wave * 64, esz = a.out_bf16 ? 2 : 4;
    pw_wait_barrier<0>();                                                    // nobody reads the rings any more
    if (c0 + (actf ? 32 : 64) <= oc && (out_ld * esz) % 16 == 0 && (uintptr_t)out_p % 16 == 0 && !(a.scatter_rows && !a.single_expert)) {
        constexpr int LD = 72;
        float* pad = reinterpret_cast<float*>(smem) + wave * (32 * LD);
        static_assert(4 * 32 * LD * 4 <= OFF_S, "in the rings");
#pragma unroll
        for (int b = 0; b < NB; b++) {
            const int left = rows - b * 32;                                  // of this block
            if (left <= 0) break;
#pragma unroll
            for (int c = 0; c < NC; c++)
#pragma unroll
                for (int i = 0; i < 16; i++) pad[((i & 3) + 8 * (i >> 2) + 4 * khalf) * LD + c * 32 + n31] = acc[b][c][i];
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront"); __builtin_amdgcn_wave_barrier(); __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
            if (actf) {
#pragma unroll 1
                for (int r0 = 0; r0 < min(left, 32); r0 += 8) {
                    const int r = r0 + (lane >> 3), c4 = (lane & 7) * 4;
                    const float rm = rmul[b * 32 + r];
                    const float4 g = *reinterpret_cast<const float4*>(pad + r * LD + c4), u = *reinterpret_cast<const float4*>(pad + r * LD + 32 + c4);
                    const float4 v = make_float4(pfh_act(a.act_fused, g.x * rm, u.x * rm, a.act_limit, a.act_alpha), pfh_act(a.act_fused, g.y * rm, u.y * rm, a.act_limit, a.act_alpha),
                                                 pfh_act(a.act_fused, g.z * rm, u.z * rm, a.act_limit, a.act_alpha), pfh_act(a.act_fused, g.w * rm, u.w * rm, a.act_limit, a.act_alpha));
                    if (r < left) *reinterpret_cast<float4*>(out_p + (size_t)(row0 + b * 32 + r) * out_ld + c0 + c4) = v;
                }
            } else if (esz == 4) {
#pragma unroll 1
                for (int r0 = 0; r0 < min(left, 32); r0 += 4) {
                    const int r = r0 + (lane >> 4), c4 = (lane & 15) * 4;
                    const float rm = rmul[b * 32 + r];
                    const float4 v = *reinterpret_cast<const float4*>(pad + r * LD + c4);
                    if (r < left) *reinterpret_cast<float4*>(out_p + (size_t)(row0 + b * 32 + r) * out_ld + c0 + c4) = make_float4(v.x * rm, v.y * rm, v.z * rm, v.w * rm);
                }
            } else {
#pragma unroll 1
                for (int r0 = 0; r0 < min(left, 32); r0 += 8) {
                    const int r = r0 + (lane >> 3), c8 = (lane & 7) * 8;
                    const float rm = rmul[b * 32 + r];
                    const float4 v0 = *reinterpret_cast<const float4*>(pad + r * LD + c8), v1 = *reinterpret_cast<const float4*>(pad + r * LD + c8 + 4);
                    const float v[8] = {v0.x * rm, v0.y * rm, v0.z * rm, v0.w * rm, v1.x * rm, v1.y * rm, v1.z * rm, v1.w * rm};
                    uint16_t h[8];
#pragma unroll
                    for (int e = 0; e < 8; e++) if (a.out_bf16 == 1) pfh_put<1>(h, e, v[e]); else pfh_put<2>(h, e, v[e]);
                    if (r < left)
                        *reinterpret_cast<u32x4*>(reinterpret_cast<uint16_t*>(out_p) + (size_t)(row0 + b * 32 + r) * out_ld + c0 + c8) =
                            u32x4{h[0] | ((uint32_t)h[1] << 16), h[2] | ((uint32_t)h[3] << 16), h[4] | ((uint32_t)h[5] << 16), h[6] | ((uint32_t)h[7] << 16)};
                }
            }
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront"); __builtin_amdgcn_wave_barrier(); __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        }
        return;
    }
#define PW_ST(OT_, A_) pfh_store_tile<NB, NC, false, OT_, A_>(acc, nsb, rows, row0, rmul, row_dst, out_p, out_ld, col, m.N, lane, a.act_fused, a.act_limit, a.act_alpha)
    if (actf) PW_ST(0, true);
    else if (a.out_bf16 == 1) PW_ST(1, false);
    else if (a.out_bf16 == 2) PW_ST(2, false);
    else PW_ST(0, false);
#undef PW_ST
}
}  // namespace

static int pfw_columns(const KrPfGemmHArgs& a) {
    int ncb = (a.m.N + BN - 1) / BN;
    for (int i = 0; i < a.n_extra; i++) ncb += (a.mx[i].N + BN - 1) / BN;
    return ncb;
}
// dense problems: where the tiles come near one a compute unit; below that kr_pfh_gemm_kernel's of 64 x 128 spread wider (us, there / here: 2752 x 2048 x 4096, 232 tiles 75 / 63, 400 x 12352 x 2048, 245
// tiles 40 / 35, but 2048 x 2048 x 4096, 176 tiles 51 / 60 and 4096 x 1024 x 2048, 172 tiles 29 / 34).  Those are launches alone.  Beside another chunk's launches the smaller problems are as well off here: whole
// prompts of 700 - 8192 tokens, the line at 170 / at 220 / never: 700 2.19 / 2.20 / 2.24 ms, 2300 3.97 / 4.03, 4096 5.92 / 5.97 / 6.2, 7000 9.01 / 9.22, 8192 10.24 / 10.38 / 11.0; at 120 as at 170.
bool kr_pfw_dense(const KrPfGemmHArgs& a) {
    if (!a.single_expert || a.m.bits != 4 || a.m.qs || a.form != KR_PFH_AUTO) return false;
    for (int i = 0; i < a.n_extra; i++) if (a.mx[i].bits != 4 || a.mx[i].qs || a.mx[i].ng != a.m.ng) return false;
    return (long)((a.total_rows + BM - 1) / BM) * pfw_columns(a) >= 220;
}
void kr_pfw_launch(const KrPfGemmHArgs& a, int mt, hipStream_t st) {
    if (mt <= 0 || kr_lds_optin((const void*)kr_pfw_gemm_kernel, LDS_BYTES)) return;      // (the caller sees the runtime's error)
    const int ncb = pfw_columns(a), span = 8 * a.run;
    const dim3 grid(a.single_expert ? 8 * ((mt * ncb + 7) / 8) : (mt + span - 1) / span * span * ncb);
    hipLaunchKernelGGL(kr_pfw_gemm_kernel, grid, dim3(256), LDS_BYTES, st, a);
}
