// The grouped products of a long prompt on A8 banks: 256 weight rows against up to 256 of an expert's rows per
// workgroup (a8_wide.hip), behind d3_moe_a8_prefill.
#pragma once
#include "wide_tile.hpp"

namespace d3 {

// 16-row tiles of a pass. FP8 takes half as many: its float32 sums are added up as the grouped products add them, K
// slice by K slice, so that a row's result does not depend on how many rows run with it, which takes a second set of
// accumulators.
__host__ __device__ constexpr int a8_wide_tiles(int format) { return format == 3 ? 8 : 16; }

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
