// A long prompt's (row, expert) pairs grouped by expert over many workgroups, with the passes of the wide products: each
// block of pairs counted by itself (prompt_hist_block), then every block's pairs dealt to their places, which the
// blocks' counts alone determine (prompt_group.hip). One workgroup's LDS atomics take 1 ns a pair, more where routing is
// skewed. Measured in a kernel trace for 32768 and 65536 pairs of 128 experts, us in one workgroup / here: even routing, A8
// banks (int32 places) 36 / 10 and 66 / 10, the reference's (int64 order and inverse) 33 / 8 and 60 / 8; Zipf(1.1) routing,
// the reference's at 65536 92 / 16, of which the counts' 5 ride with the rows' planes on int8, W4 and W6.
#pragma once
#include "wide_tile.hpp"

namespace d3 {

constexpr int PG_BLOCKS = 64;      // at most, per prompt
constexpr int PG_MAX_E = 1024;

struct PromptGroups {
  const int64_t* ids;          // [P]
  int P, E;
  bool clamp;                  // ids outside [0, E): the nearest expert, else after every group with inverse -1
  int64_t* order = nullptr;    // [P] place -> pair, or perm
  int* perm = nullptr;
  int* inverse = nullptr;      // [P] pair -> place, or null
  int* count;                  // passes listed
  int4* passes;                // [cap] (expert, first place, rows, 0), the passes with most tiles first
  int cap, tiles;              // at most `tiles` 16-row tiles a pass
  int* hist;                   // [PG_BLOCKS, E]
};

// pairs per block: whole workgroups' worth, at most PG_BLOCKS of them
__host__ __device__ inline int pg_block(int P) {
  const int per = (P + PG_BLOCKS - 1) / PG_BLOCKS;
  return per < 1024 ? 1024 : (per + 255) / 256 * 256;
}
__host__ __device__ inline int pg_blocks(int P) { return (P + pg_block(P) - 1) / pg_block(P); }

// hist[b] = the experts' counts in block b of the pairs; a workgroup of any size, cnt E words of LDS
D3_INLINE void prompt_hist_block(const PromptGroups& g, int b, int* cnt) {
  for (int e = threadIdx.x; e < g.E; e += blockDim.x) cnt[e] = 0;
  __syncthreads();
  const int from = b * pg_block(g.P), to = min(g.P, from + pg_block(g.P));
  for (int p = from + threadIdx.x; p < to; p += blockDim.x) {
    int64_t e = g.ids[p];
    if (g.clamp) e = min<int64_t>(max<int64_t>(e, 0), g.E - 1);
    if (e >= 0 && e < g.E) atomicAdd(&cnt[e], 1);
  }
  __syncthreads();
  for (int e = threadIdx.x; e < g.E; e += blockDim.x) g.hist[(size_t)b * g.E + e] = cnt[e];
}

void launch_prompt_hist(const PromptGroups& g, hipStream_t s);
void launch_prompt_scatter(const PromptGroups& g, hipStream_t s);

}  // namespace d3
