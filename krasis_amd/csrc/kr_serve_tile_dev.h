// kr_serve_tile_dev.h -- what the prompt tiles of the serving step share: rows of a slot, the LDS-DMA request, the wait that ends a slot.
#ifndef KR_SERVE_TILE_DEV_H
#define KR_SERVE_TILE_DEV_H
#include "kr_serve_gemm_dev.h"

constexpr int TL_ROW = 128;                                    // bytes of a slot's row, whole cache lines (rows of 64 bytes fetch every line twice): 64 k in bf16, 32 in f32

__device__ __forceinline__ uint32_t tl_lds_addr(const void* p) { return (uint32_t)(uintptr_t)(const __attribute__((address_space(3))) char*)p; }
// 64 lanes x 16 bytes from the lane's own address to lds_dst (wave-uniform) + 16 lane.  M0 is the compiler's register: saved and restored inside.  The compiler
// does not count this request; the waits below do.
__device__ __forceinline__ void tl_dma16(uint32_t lds_dst, const void* src) {
    unsigned keep;
    asm volatile("s_mov_b32 %0, m0\n\ts_mov_b32 m0, %2\n\ts_nop 2\n\tglobal_load_lds_dwordx4 %1, off\n\ts_mov_b32 m0, %0" : "=&s"(keep) : "v"(src), "s"(lds_dst) : "memory");
}
// at most N of this wave's requests are outstanding and its LDS reads have returned, then the workgroup barrier
template <int N> __device__ __forceinline__ void tl_wait_barrier() { asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" :: "n"(N) : "memory"); }

void kr_sv_gemm_tile_f32(const KrSvGemm& g, hipStream_t st);   // kr_serve_tile_f32.hip
#endif
