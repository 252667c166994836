// The grouped products of a long prompt on FP8 banks in the reference's layout (e4m3 with a float scale per 128 x 128
// block), held whole on the GPU: what grouped_fp8_kernel computes (exact bf16 planes of the rows, exact bf16 weights,
// float32 sums of each 128-column block scaled and added up), for prompts whose experts have many rows each.
//
// grouped_fp8_kernel reads and widens every weight again per 32 rows. Here a workgroup runs 256 weight rows against up
// to 96 rows: the weights lie in LDS as their e4m3 bytes, 128 columns at a time, and each wave widens its 64 rows'
// operands as it reads them (two codes an instruction); the rows lie there as bf16, in tiles of 64 columns. A lane's
// columns of 128 are grouped_fp8_kernel's, 32 (l >> 4) .. + 31 in four steps of 8, weights and rows alike, and the planes
// meet in its order, so that a row's float32 sums are the same however many rows run with it.
// Measured us per layer, 32-row / here: 8192 rows, top-8 of 128 experts (FFN 768, Zipf routing) 2266 / 1352 (in a kernel
// trace the first bank's products 1196 / 560, the second's, three planes, 966 / 752), 2391 rows of 256 experts (FFN 512)
// 625 / 414. (With the columns in memory order, whole 128-byte lines a copy, 1331 and 408: other sums at other lengths.)
#include "ref_common.hpp"
#include "wide_tile.hpp"
#include "../../include/drama3_moe.h"

#include <algorithm>
#include <string>

namespace d3 {
int fail(const std::string& msg);
int hip_fail(hipError_t err, const char* what);
namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
constexpr int WF_W = WT_N * 128;                // 128 columns of the weights
constexpr int WF_X = 16 * WIDE_TILES * 128;     // 64 columns of a pass's rows, one plane
constexpr int WF_CHUNKS = 16;                   // K <= 2048

struct WideF8Args {
  const uint8_t* xs;    // bf16 planes [PL][plane]
  int64_t plane;        // bytes
  const int64_t* order;
  int k_order, xrows;
  const int* count;
  const int4* passes;   // (expert, first row, rows, 0)
  const uint8_t* w;     // [E * N, K]
  const float* s;       // [E * N / 128, K / 128]
  float* out;           // [rows, N], or [rows, N / 2] with SwiGLU
  int N, K;
};

// eight e4m3 codes as bf16, exactly
D3_INLINE bf16x8 widen8(uint32_t lo, uint32_t hi) {
  typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
  const bf16x2 a = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(lo, 1.0f, false);
  const bf16x2 b = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(lo, 1.0f, true);
  const bf16x2 c = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(hi, 1.0f, false);
  const bf16x2 d = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(hi, 1.0f, true);
  return bf16x8{a[0], a[1], b[0], b[1], c[0], c[1], d[0], d[1]};
}

// A stage is 128 columns of one plane (bf16 rows as they are), or of three planes two of the four steps: columns 32 j +
// 16 (s & 1) .. + 15, j < 4, of 128 in stage s. SWIGLU as wide_i8_kernel's.
template <int PL, bool SWIGLU>
__global__ void __launch_bounds__(WT_THREADS, 2) wide_fp8_kernel(WideF8Args a) {
  constexpr int TP = PL == 1 ? 2 : 3;      // tiles of 64 columns per row and stage: the halves, or the planes
  constexpr int HALVES = PL == 1 ? 2 : 1;  // of 128 columns, per stage
  constexpr int COPIES = (12 * TP + 7) / 8;
  __shared__ __attribute__((aligned(1024))) uint8_t smem[2 * (WF_W + TP * WF_X)];
  __shared__ float bscale[2][WF_CHUNKS];
  const int N = a.N, K = a.K, chunks = K / 128, stages = chunks * 2 / HALVES;
  int pass, xb;
  wt_place(blockIdx.x, N / WT_N, pass, xb);
  if (pass >= a.count[0]) return;
  const int4 p4 = a.passes[pass];
  const int expert = __builtin_amdgcn_readfirstlane(p4.x), first = __builtin_amdgcn_readfirstlane(p4.y),
            rows = __builtin_amdgcn_readfirstlane(p4.z), tiles = (rows + 15) / 16;
  const int tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int q = lane >> 4, c = lane & 15, wn = w & 3, wm = w >> 2;
  const size_t n0 = (size_t)expert * N + (size_t)xb * (SWIGLU ? WT_N / 2 : WT_N);
  auto bank_row = [&](int block) { return SWIGLU ? 32 * (block >> 1) + (block & 1) * (N / 2) : 32 * block; };
  const uint32_t lds0 = lds_address(smem), ldsx = lds0 + 2 * WF_W;
  // the workgroup's two row blocks' scales: rows n0 .. + 127, and the next 128 (SwiGLU: the up rows)
  if (tid < 2 * chunks) {
    const int blk = tid >= chunks, ch = tid - blk * chunks;
    bscale[blk][ch] = a.s[((n0 + (blk ? (SWIGLU ? N / 2 : 128) : 0)) / 128) * chunks + ch];
  }

  // the rows: 12 blocks of 8 rows x TP tiles, dealt to the waves as wide_i8_kernel's planes
  uint32_t xoff[3];
  {
    int p[3];
#pragma unroll
    for (int i = 0; i < 3; i++) p[i] = first + min(8 * ((w + 8 * i) % 12) + (lane >> 3), rows - 1);
    if (a.order) {
#pragma unroll
      for (int i = 0; i < 3; i++) p[i] = (int)a.order[p[i]];
#pragma unroll
      for (int i = 0; i < 3; i++) p[i] = pair_row(p[i], a.k_order, a.xrows);
    }
#pragma unroll
    for (int i = 0; i < 3; i++) {
      const int piece = wt_slot(8 * ((w + 8 * i) % 12) + (lane >> 3), lane & 7);
      xoff[i] = (uint32_t)p[i] * (uint32_t)(2 * K) + (PL == 1 ? 16 * piece : 64 * (piece >> 1) + 16 * (piece & 1));
    }
  }
  auto load_rows = [&](int stage, int i) __attribute__((always_inline)) {  // copy i < COPIES of this wave
    const int n = w + 8 * i, b = n % 12, t = n / 12;
    if (n < 12 * TP && (b >> 1) < tiles)
      dma16(ldsx + (uint32_t)((stage & 1) * TP * WF_X + t * WF_X + b * 1024),
            a.xs + (PL == 1 ? 256 * (int64_t)stage + 128 * t : t * a.plane + 256 * (int64_t)(stage >> 1) + 32 * (stage & 1)),
            xoff[i % 3]);
  };
  uint32_t woff[2];
#pragma unroll
  for (int i = 0; i < 2; i++) {
    const int r = 8 * i + (lane >> 3);
    woff[i] = (uint32_t)(r * K) + 16 * wt_slot(r, lane & 7);
  }
  const uint8_t* wwave = a.w + (n0 + bank_row(w)) * K;
  auto load_weights = [&](int chunk, int i) __attribute__((always_inline)) {  // copy i < 4 of this wave
    dma16(lds0 + (chunk & 1) * WF_W + w * 4096 + 1024 * i, wwave + 128 * chunk + (size_t)(i >> 1) * 16 * K, woff[i & 1]);
  };
#pragma unroll
  for (int i = 0; i < COPIES; i++) load_rows(0, i);
#pragma unroll
  for (int i = 0; i < 4; i++) load_weights(0, i);

  auto run = [&]<int NT>() __attribute__((always_inline)) {
    f32x4 acc[NT][4], part[NT][4];  // the sums, and the present 128 columns' before their block scale
#pragma unroll
    for (int j = 0; j < NT; j++)
#pragma unroll
      for (int n = 0; n < 4; n++) acc[j][n] = part[j][n] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    i32x4 raw[4];
    bf16x8 b[2][PL][2];
    int at[HALVES][2];  // step 2 h + u of the stage: piece 4 q + 2 h + u of a plane's two tiles, or 2 q + u of its one
#pragma unroll
    for (int h = 0; h < HALVES; h++)
#pragma unroll
      for (int u = 0; u < 2; u++)
        at[h][u] = c * 128 + (PL == 1 ? (q >> 1) * WF_X + 16 * wt_slot(c, 4 * (q & 1) + 2 * h + u) : 16 * wt_slot(c, 2 * q + u));
    auto read_w = [&](int chunk, int h) __attribute__((always_inline)) {  // steps 2 h and 2 h + 1 of the chunk
      const uint8_t* src = smem + (chunk & 1) * WF_W + (64 * wn) * 128 + c * 128 + 16 * wt_slot(c, 2 * q + h);
#pragma unroll
      for (int n = 0; n < 4; n++) raw[n] = *(const i32x4*)(src + n * 2048);
    };
    auto read_x = [&](int stage, int h, int j, bf16x8 (&v)[PL][2]) __attribute__((always_inline)) {
      const uint8_t* src = smem + 2 * WF_W + (stage & 1) * TP * WF_X + (wm + 2 * j) * 2048;
#pragma unroll
      for (int t = 0; t < PL; t++)
#pragma unroll
        for (int u = 0; u < 2; u++) v[t][u] = *(const bf16x8*)(src + (PL == 1 ? 0 : t) * WF_X + at[h][u]);
    };
    dma_wait();
    __syncthreads();
    for (int s = 0; s < stages; s++) {
      const bool more = s + 1 < stages;
      const int chunk = PL == 1 ? s : s >> 1;
      // three planes: the chunk's weights were read with its first stage's; this stage's half of them
      read_w(chunk, PL == 1 ? 0 : s & 1);
      read_x(s, 0, 0, b[0]);
      if (more) {
#pragma unroll
        for (int i = 0; i < COPIES; i++) load_rows(s + 1, i);
        if (PL == 1 || ((s & 1) == 0 && chunk + 1 < chunks)) {
#pragma unroll
          for (int i = 0; i < 4; i++) load_weights(chunk + 1, i);
        }
      }
#pragma unroll
      for (int h = 0; h < HALVES; h++) {
        bf16x8 wa[4][2];
#pragma unroll
        for (int n = 0; n < 4; n++) {
          wa[n][0] = widen8((uint32_t)raw[n].x, (uint32_t)raw[n].y);
          wa[n][1] = widen8((uint32_t)raw[n].z, (uint32_t)raw[n].w);
        }
        if (h + 1 < HALVES) read_w(chunk, h + 1);
#pragma unroll
        for (int j = 0; j < NT; j++) {
          const int cur = (h * NT + j) & 1;
          if (j + 1 < NT) read_x(s, h, j + 1, b[cur ^ 1]);
          else if (h + 1 < HALVES) read_x(s, h + 1, 0, b[cur ^ 1]);
          __builtin_amdgcn_sched_barrier(0);  // the reads first
#pragma unroll
          for (int u = 0; u < 2; u++)
#pragma unroll
            for (int t = 0; t < PL; t++)
#pragma unroll
              for (int n = 0; n < 4; n++)
                part[j][n] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wa[n][u], b[cur][t][u], part[j][n], 0, 0, 0);
          __builtin_amdgcn_sched_barrier(0);
        }
      }
      if (PL == 1 || (s & 1)) {
        const float s0 = bscale[SWIGLU ? 0 : wn >> 1][chunk], s1 = bscale[SWIGLU ? 1 : wn >> 1][chunk];
#pragma unroll
        for (int j = 0; j < NT; j++)
#pragma unroll
          for (int n = 0; n < 4; n++) {
#pragma unroll
            for (int i = 0; i < 4; i++) acc[j][n][i] = fmaf(n < 2 ? s0 : s1, part[j][n][i], acc[j][n][i]);
            part[j][n] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
          }
      }
      dma_wait();
      __syncthreads();
    }
    // lane l holds weight rows 64 wn + 16 n + 4 q .. + 3 of the pass's row 16 (wm + 2 j) + c
#pragma unroll
    for (int j = 0; j < NT; j++) {
      const int r = 16 * (wm + 2 * j) + c;
      if (r < rows) {
        if constexpr (SWIGLU) {
          float* o = a.out + (size_t)(first + r) * (N / 2) + xb * (WT_N / 2) + 32 * wn + 4 * q;
#pragma unroll
          for (int n = 0; n < 2; n++) {
            f32x4 h;
#pragma unroll
            for (int i = 0; i < 4; i++) h[i] = silu_up(acc[j][n][i], acc[j][n + 2][i]);
            *(f32x4*)(o + 16 * n) = h;
          }
        } else {
          float* o = a.out + (size_t)(first + r) * N + xb * WT_N + 64 * wn + 4 * q;
#pragma unroll
          for (int n = 0; n < 4; n++) *(f32x4*)(o + 16 * n) = acc[j][n];
        }
      }
    }
  };
  switch ((tiles - wm + 1) / 2) {  // (a wave without a tile runs the operands of one and stores nothing)
    case 3: run.template operator()<3>(); break;
    case 2: run.template operator()<2>(); break;
    default: run.template operator()<1>(); break;
  }
}

}  // namespace
}  // namespace d3

using namespace d3;

extern "C" int d3_prompt_fp8(const void* planes, int32_t n_planes, int64_t plane, const int64_t* order, int32_t k,
                             int32_t rows, const int32_t* passes, int64_t pass_ints, int32_t E, const void* w,
                             const float* s, float* out, int32_t N, int32_t K, int32_t swiglu, void* stream) {
  if (!planes || !passes || !w || !s || !out) return fail("d3_prompt_fp8: null pointer");
  if (n_planes != 1 && n_planes != 3) return fail("d3_prompt_fp8: 1 or 3 planes");
  if (N < WT_N || N % WT_N || K < 256 || K % 256 || K > 2048) return fail("d3_prompt_fp8: N % 256 == 0, K % 256 == 0, K <= 2048");
  if (plane < K || plane % K || 2 * plane > (int64_t)UINT32_MAX - 4096) return fail("d3_prompt_fp8: plane a multiple of K, under 2^32 bytes");
  if (rows < 1 || E < 1 || (order ? k < 1 : rows > plane / K))
    return fail("d3_prompt_fp8: 1 <= rows (<= plane / K without order), k >= 1 with order");
  if (((uintptr_t)planes | (uintptr_t)w) & 15) return fail("d3_prompt_fp8: planes and weights at 16-byte alignment");
  if (pass_ints < d3_prompt_pass_ints(E, rows)) return fail("d3_prompt_fp8: passes holds fewer than d3_prompt_pass_ints ints");
  const int cap = rows / (16 * WIDE_TILES) + std::min(E, rows);
  WideF8Args a;
  a.xs = (const uint8_t*)planes;
  a.plane = 2 * plane;
  a.order = order;
  a.k_order = k;
  a.xrows = (int)(plane / K);
  a.count = passes;
  a.passes = (const int4*)(passes + 4);
  a.w = (const uint8_t*)w;
  a.s = s;
  a.out = out;
  a.N = N;
  a.K = K;
  const dim3 grid((unsigned)(wt_places(cap) * (N / WT_N)));
  const hipStream_t st = (hipStream_t)stream;
  if (n_planes == 1) {
    if (swiglu) hipLaunchKernelGGL((wide_fp8_kernel<1, true>), grid, dim3(WT_THREADS), 0, st, a);
    else hipLaunchKernelGGL((wide_fp8_kernel<1, false>), grid, dim3(WT_THREADS), 0, st, a);
  } else {
    if (swiglu) hipLaunchKernelGGL((wide_fp8_kernel<3, true>), grid, dim3(WT_THREADS), 0, st, a);
    else hipLaunchKernelGGL((wide_fp8_kernel<3, false>), grid, dim3(WT_THREADS), 0, st, a);
  }
  const hipError_t e = hipGetLastError();
  return e == hipSuccess ? 0 : hip_fail(e, "d3_prompt_fp8");
}
