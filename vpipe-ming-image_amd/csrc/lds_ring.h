// What the projection kernels' LDS rings share: global->LDS DMA as inline
// asm, the ring's explicit wait, the bank swizzles and the tile order.
#pragma once

#include "common.h"

namespace ming {

// LDS swizzles for gfx950's 64 x 4-byte banks: a ds_read_b128 serves 16
// lanes (256 B) per cycle, and a fragment read has those 16 lanes on 16
// consecutive rows at one logical chunk. Rows of 128 B (8 chunks) pair up
// per 256-B bank line, so the chunk is XORed with (row >> 1) & 7; rows of
// 64 B (4 chunks) fill a line four at a time: XOR with (row >> 2) & 3.
__device__ __forceinline__ int swz8(int row, int c) { return row * 8 + (c ^ ((row >> 1) & 7)); }
__device__ __forceinline__ int swz4(int row, int c) { return row * 4 + (c ^ ((row >> 2) & 3)); }

// The DMA written as inline asm, for rings whose waits are all
// explicit: the compiler then sees no LDS store it must order reads
// against, so it cannot add a drain of its own (its alias tracking of LDS
// DMA gives up at loop joins and would wait for vmcnt(0)). M0 carries the
// wave's LDS byte address; the s_nop covers the M0 -> LDS-DMA hazard.
// Correctness rests on the ring's own waits: ring_wait<N>() below, which
// also orders every LDS access against the DMAs through its memory clobber.
#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"
// Scalar-base form: address = 64-bit wave-uniform base (SGPRs) + 32-bit
// per-lane byte offset, so advancing a stage is a scalar add and the issue
// needs no VALU address arithmetic.
__device__ __forceinline__ void dma16_sb(const void* base, uint32_t off, uint32_t lds) {
  asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1"
               :: "v"(off), "s"(base), "s"(lds) : "m0");
}
__device__ __forceinline__ void dma4_sb(const void* base, uint32_t off, uint32_t lds) {
  asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dword %0, %1"
               :: "v"(off), "s"(base), "s"(lds) : "m0");
}
#pragma clang diagnostic pop

// LDS byte address of a __shared__ object: the low half of its generic
// address is the offset inside the workgroup's LDS.
__device__ __forceinline__ uint32_t lds_addr(const void* p) {
  return static_cast<uint32_t>(reinterpret_cast<uintptr_t>(p));
}

// Ring barrier with its vmcnt: this wave's DMAs except the newest N have
// landed, its LDS reads are complete, then the workgroup barrier. After it
// every wave's older DMAs are visible and every wave is done reading.
template <int N>
__device__ __forceinline__ void ring_wait() {
  static_assert(N >= 0 && N < 64, "vmcnt field is 6 bits");
  asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" :: "n"(N) : "memory");
}

// Logical tile of a block: each XCD a contiguous range of the tile grid,
// walked in a grouped raster of 4 tile-rows.
__device__ __forceinline__ void tile_of_block(int b, int tiles_m, int tiles_n,
                                              int* tm, int* tn) {
  const int nb = tiles_m * tiles_n;
  const int q = nb / 8, rem = nb % 8;
  const int xcd = b % 8, local = b / 8;
  const int v = xcd * q + (xcd < rem ? xcd : rem) + local;
  constexpr int GM = 4;
  const int gsz = GM * tiles_n;
  const int g = v / gsz;
  const int first = g * GM;
  const int gm = (tiles_m - first) < GM ? (tiles_m - first) : GM;
  const int r = v - g * gsz;
  *tm = first + r % gm;
  *tn = r / gm;
}

}  // namespace ming
