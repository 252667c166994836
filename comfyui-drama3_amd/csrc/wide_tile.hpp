// The wide tile of the prompt products: what the kernels share that run 256 weight rows against many of an expert's
// rows. Both operands of a 128-column stage sit in LDS as rows of 128 bytes, in 16-byte pieces: piece j of row r at
// slot j ^ ((r >> 1) & 7). A wave's copy of 8 rows (lane l: slot l & 7 of row l >> 3) then reads each row's 128 bytes
// from memory as one line, and a 16 x 16 x 64 MFMA operand (lane l: row l & 15, piece 4 half + (l >> 4)) reads 16
// different 16-byte banks per 16 lanes, without conflicts. (Stages of 64 columns through a ring of four places, two
// stages on their way, measured 10% slower on int8: twice the barriers, and half lines from L2.)
#pragma once
#include "common.hpp"

namespace d3 {

constexpr int WT_N = 256;       // weight rows per workgroup
constexpr int WT_THREADS = 512; // 8 waves: 4 over the weight rows (64 each), 2 over the expert's rows (tiles in turn)
constexpr int WIDE_TILES = 6;   // 16-row tiles of a pass over three int8 planes
constexpr int WT_CHUNK = 4;     // passes an XCD takes together (one after the other in the list)

// LDS byte address of a shared object
D3_INLINE uint32_t lds_address(const void* p) {
  return (uint32_t)(uintptr_t)(__attribute__((address_space(3))) const void*)p;
}
// 16 bytes per lane from base + off (the lane's own) into LDS at lds + 16 * lane (lds uniform over the wave), without
// passing through registers. The instruction takes lds from m0: as an operand of the statement, so that the compiler
// knows what m0 holds after it. A scalar register that a vector instruction wrote (readfirstlane) may be read by a memory
// instruction five wait states later at the earliest: the hardware does not wait, and the compiler, which inserts an
// s_nop 4 there before loads of its own, does not look into the statement. A scalar instruction may read it at once, and
// what that writes may be read at once: the base goes through an s_mov (with an s_nop 4 in its place 8192 W6 rows took
// 0.6% longer), which is also the one wait state between setting m0 and the copy. The compiler does not count these
// loads: dma_wait() before the barrier that hands them to the other waves.
D3_INLINE void dma16(uint32_t lds, const void* base, uint32_t off) {
  // (both uniform already; said again for the compiler, which may keep a loop's pointers in vector registers)
  const uint64_t at = (uint64_t)base;
  const uint64_t sbase = (uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)at) |
                         (uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((int)(at >> 32)) << 32;
  uint64_t from;
  asm volatile("s_mov_b64 %0, %3\n\tglobal_load_lds_dwordx4 %2, %0"
               : "=&s"(from)
               : "{m0}"(__builtin_amdgcn_readfirstlane((int)lds)), "v"(off), "s"(sbase)
               : "memory");
}
D3_INLINE void dma_wait() { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); }

// the slot of 16-byte piece j of row r
D3_INLINE int wt_slot(int r, int j) { return j ^ ((r >> 1) & 7); }

// The pass and the 256-row column of a workgroup: workgroup i of a launch runs on XCD i % 8; WT_CHUNK passes that
// follow each other in the list (mostly one expert's) go to one XCD with all nx columns of each, so that their weight
// rows and their planes are read once into that XCD's L2.
D3_INLINE void wt_place(int lin, int nx, int& pass, int& xb) {
  const int xcd = lin & 7, k = lin >> 3, per = WT_CHUNK * nx, r = k % per;
  pass = ((k / per) * 8 + xcd) * WT_CHUNK + r % WT_CHUNK;
  xb = r / WT_CHUNK;
}
__host__ __device__ constexpr int wt_places(int cap) { return (cap + 8 * WT_CHUNK - 1) / (8 * WT_CHUNK) * (8 * WT_CHUNK); }

// An expert's n rows as passes of at most `most` 16-row tiles, all with the same number of tiles but the last.
D3_INLINE int wt_passes(int n, int most) { return ((n + 15) / 16 + most - 1) / most; }
D3_INLINE int wt_tiles(int n, int most) {
  const int t = (n + 15) / 16, p = (t + most - 1) / most;
  return p ? (t + p - 1) / p : 0;
}

}  // namespace d3
