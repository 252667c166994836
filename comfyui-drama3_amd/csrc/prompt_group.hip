// A long prompt's pairs grouped by expert (offload.py:140-143's sort and counts), see prompt_group.hpp: two launches,
// the blocks' counts and the dealing.
#include "prompt_group.hpp"

namespace d3 {
namespace {

__global__ void __launch_bounds__(1024) prompt_hist_kernel(PromptGroups g) {
  __shared__ int cnt[PG_MAX_E];
  prompt_hist_block(g, blockIdx.x, cnt);
}

// Workgroup b deals block b's pairs: each expert's first place (the sum of the smaller experts' pairs) and the pairs of
// its earlier blocks, both from hist, then an LDS counter per expert. Workgroup 0 also lists the passes. Within a block
// the pairs' order is that of their atomic adds: every output row depends on its own pair alone.
__global__ void __launch_bounds__(1024) prompt_scatter_kernel(PromptGroups g) {
  __shared__ int total[PG_MAX_E], before[PG_MAX_E], cursor[PG_MAX_E + 1], wave_total[16], pcount[16], pcursor[16], seen;
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6, E = g.E, b = blockIdx.x, blocks = gridDim.x;
  total[tid] = 0;
  before[tid] = 0;
  if (tid < 16) pcount[tid] = 0;
  if (tid == 0) seen = 0;
  __syncthreads();
  int span = 64;  // threads per run over the experts: E rounded up to a power of two
  while (span < E) span <<= 1;
  const int e = tid & (span - 1);
  int mine = 0;  // pairs of expert e in earlier blocks, by this thread's share of them
  if (e < E) {
    int all = 0;
#pragma unroll 8
    for (int i = tid / span; i < blocks; i += 1024 / span) {
      const int h = g.hist[(size_t)i * E + e];
      all += h;
      mine += i < b ? h : 0;
    }
    atomicAdd(&total[e], all);
    atomicAdd(&before[e], mine);
  }
  mine = wave_sum_i32(mine);
  if (lane == 0) atomicAdd(&seen, mine);
  __syncthreads();
  // exclusive prefix of the totals, thread t expert t
  const int v = tid < E ? total[tid] : 0;
  int incl = v;
#pragma unroll
  for (int d = 1; d < 64; d <<= 1) {
    const int u = __shfl_up(incl, d);
    if (lane >= d) incl += u;
  }
  if (lane == 63) wave_total[w] = incl;
  __syncthreads();
  int earlier = 0, everything = 0;
  for (int i = 0; i < 16; i++) {
    if (i < w) earlier += wave_total[i];
    everything += wave_total[i];
  }
  const int first = earlier + incl - v;
  if (tid < E) cursor[tid] = first + before[tid];
  // ids outside the experts come last; this block's follow those of the blocks before it
  if (tid == 0) cursor[E] = everything + (b * pg_block(g.P) - seen);
  __syncthreads();
  const int from = b * pg_block(g.P), to = min(g.P, from + pg_block(g.P));
  for (int p = from + tid; p < to; p += 1024) {
    int64_t id = g.ids[p];
    if (g.clamp) id = min<int64_t>(max<int64_t>(id, 0), E - 1);
    const bool valid = id >= 0 && id < E;
    const int at = atomicAdd(&cursor[valid ? (int)id : E], 1);
    if (g.order) g.order[at] = p;
    else g.perm[at] = p;
    if (g.inverse) g.inverse[p] = valid ? at : -1;
  }
  if (b == 0) {  // bucket k: passes of tiles - k tiles
    const int np = wt_passes(v, g.tiles), tiles = wt_tiles(v, g.tiles);
    if (np) atomicAdd(&pcount[g.tiles - tiles], np);
    __syncthreads();
    if (tid == 0) {
      int at = 0;
      for (int k = 0; k < g.tiles; k++) {
        pcursor[k] = at;
        at += pcount[k];
      }
      g.count[0] = min(at, g.cap);
    }
    __syncthreads();
    if (np) {
      const int at = atomicAdd(&pcursor[g.tiles - tiles], np), step = 16 * tiles;
      for (int i = 0; i < np && at + i < g.cap; i++)
        g.passes[at + i] = int4{tid, first + i * step, min(step, v - i * step), 0};
    }
  }
}

}  // namespace

void launch_prompt_hist(const PromptGroups& g, hipStream_t s) {
  hipLaunchKernelGGL(prompt_hist_kernel, dim3(pg_blocks(g.P)), dim3(1024), 0, s, g);
}
void launch_prompt_scatter(const PromptGroups& g, hipStream_t s) {
  hipLaunchKernelGGL(prompt_scatter_kernel, dim3(pg_blocks(g.P)), dim3(1024), 0, s, g);
}

}  // namespace d3
