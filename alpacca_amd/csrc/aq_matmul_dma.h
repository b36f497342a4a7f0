// aq_matmul_dma.h - DMA into LDS for the matmul tile kernels.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace aq {

// 16 bytes per lane from base + voff (per lane) to LDS bytes lds + 16 * lane.
// Written in assembly because the compiler makes every later LDS read wait
// for the whole of an LDS DMA it knows of; the kernels wait themselves
// (dma_barrier) before the barrier that publishes a stage.  There are no
// output registers, and the address registers are read at issue.  M0 (the LDS
// base) has no other user in these kernels.
__device__ __forceinline__ void dma16(uint32_t lds, uint32_t voff, const void *base) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2"
               :
               : "s"(lds), "v"(voff), "s"(base)
               : "memory");
}
// 4 bytes per lane
__device__ __forceinline__ void dma4(uint32_t lds, uint32_t voff, const void *base) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dword %1, %2"
               :
               : "s"(lds), "v"(voff), "s"(base)
               : "memory");
}
// all but the last LEFT of this wave's DMAs have landed, its LDS reads are
// done, and so are those of every other wave of the workgroup
template <int LEFT>
__device__ __forceinline__ void dma_barrier() {
  asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" : : "n"(LEFT) : "memory");
}
__device__ __forceinline__ uint32_t lds_offset(const uint8_t *p) {
  return (uint32_t)(size_t)(const __attribute__((address_space(3))) uint8_t *)p;
}
template <class V>
__device__ __forceinline__ V lds_read(const uint8_t *p) {
  return *reinterpret_cast<const V *>(p);
}

// The tile of workgroup `id` (grid: tiles rounded up to a multiple of 8), or
// false past the last one.  XCD x (id modulo 8) takes a contiguous run of
// tiles, in blocks of four M tiles times all N tiles, M tiles first: the
// workgroups of an XCD share X rows and weights in its L2 (Q4_K 16384 x 2048
// at M = 2048: 272 us with all M tiles of an N tile in a row, 263 in blocks
// of four).
__device__ __forceinline__ bool xcd_tile(int id, int m_tiles, int n_tiles, int &mt, int &nt) {
  const int tiles = m_tiles * n_tiles, per_xcd = (tiles + 7) / 8;
  const int t = (id & 7) * per_xcd + (id >> 3);
  if ((id >> 3) >= per_xcd || t >= tiles) return false;
  const int tb = t / (4 * n_tiles), rest = t - tb * 4 * n_tiles;
  const int w = m_tiles - 4 * tb < 4 ? m_tiles - 4 * tb : 4;
  mt = 4 * tb + rest % w;
  nt = rest / w;
  return true;
}

}  // namespace aq
