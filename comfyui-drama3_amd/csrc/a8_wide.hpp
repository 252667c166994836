// The grouped products of a long prompt on A8 banks: 256 or 128 weight rows against up to 256 or 128 of an expert's rows
// per workgroup (a8_wide.hip), behind d3_moe_a8_prefill.
#pragma once
#include "wide_tile.hpp"

namespace d3 {

// 16-row tiles of a pass, and the weight rows of a workgroup (two threads each). int8's sums are exact; the others' float32
// sums are added up as the grouped products add them, K slice by K slice, so that a row's result does not depend on how
// many rows run with it. That takes a second set of accumulators, and half the rows. W4 and W6 (formats 1 and 2) also take
// half the weight rows, which puts two workgroups on a CU.
__host__ __device__ constexpr int a8_wide_tiles(int format) { return format == 0 ? 16 : 8; }
__host__ __device__ constexpr int a8_wide_cols(int format) { return format == 1 || format == 2 ? 128 : 256; }

struct A8WideArgs {
  const uint8_t* act;      // gate_up: the token rows [T, K]; down: the hidden rows [P, K] by sorted position
  const float* act_scale;  // gate_up: [T]; down: [P], the hidden row's scale times its routing weight
  const int* perm;         // [P] sorted position -> pair
  int k;                   // pairs per token
  const int* count;        // passes
  const int4* passes;      // (expert, first position, rows, 0)
  const uint8_t* w;        // [E * N, row bytes]
  const uint16_t* s;       // bf16 row scales [E * N], or group scales [E * N, K / 128]
  float* out;              // gate_up: SiLU(gate) * up [P, N / 2] by sorted position; down: [P, N] by pair
  int N, K;
};

// the products of one bank (down: N output rows; else N / 2 gate rows, then N / 2 up rows) over at most `cap` passes
void launch_a8_wide(int format, bool down, const A8WideArgs& a, int cap, hipStream_t s);

}  // namespace d3
