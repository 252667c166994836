// The grouped products of a long prompt on banks in the reference's integer layouts (int8 ConvRot, W4A8 and W6A8
// codes), held whole on the GPU: what grouped_i8_kernel computes (the same int8 planes, exact int32 sums and epilogue),
// for prompts whose experts have many rows each.
//
// grouped_i8_kernel takes 32 rows a pass: every pass reads and decodes its weight rows again, and each wave's 16 or 32
// weight rows read all of the pass's planes from LDS; the matrix cores were busy 10 to 20% of the time. Here a
// workgroup runs 256 weight rows against up to 96 rows (288 plane rows), a wave 64 x 48 (x 3 planes): 144 accumulators
// a lane, which still leaves two waves per SIMD, and a weight is read from L2 and decoded once per 96 rows.
// Measured, 8192 rows, top-8 of 128 experts (FFN 768, Zipf routing), both banks' products in a kernel trace, 32-row / here:
// int8 1849 / 1148 us, W4 2361 / 1383, W6 3317 / 1640; the layer untraced 1983 / 1253, 2430 / 1455, 3378 / 1695. int8's
// products alone (no copies, no stores) take 417 us of the first bank's 632 and the copies alone 364: what is left is L2
// misses that one stage ahead does not cover, and the stores (dn: 537 MB of float32). W6 adds its decoding, about 85
// vector instructions per 16 codes and pass. (The planes' sums by divisions, as the 32-row products', take 1% of a layer.)
#include "ref_common.hpp"
#include "wide_tile.hpp"
#include "../../include/drama3_moe.h"

#include <algorithm>
#include <string>

namespace d3 {
int fail(const std::string& msg);
int hip_fail(hipError_t err, const char* what);

constexpr int WI_TILES = WIDE_TILES, WI_PLANES = 3;                 // 96 rows, three planes each
constexpr int WI_W_BYTES = WT_N * 128;                              // a stage's weights
constexpr int WI_STAGE = WI_W_BYTES + WI_TILES * WI_PLANES * 2048;  // and the planes of its rows

struct WideArgs {
  const int8_t* xs;       // planes [3, plane]
  int64_t plane;
  const float* xscale;
  const int64_t* order;
  int k_order, xrows;
  const int* count;       // passes
  const int4* passes;     // (expert, first row, rows, 0)
  const uint8_t* w;       // [E * N, row bytes]
  const void* s;          // int8: row scales; codes: e4m3 group scales [E * N, K / 16]
  const float* c;         // codes: channel scales
  const float* codebook;
  float* out;             // [rows, N], or [rows, N / 2] with SwiGLU
  int N, K;
};

// W6: a 16-code group as int8-grid bytes in column order, as w6_group_i8 (clamp(rint((code - 32) * s), +-127)), two
// codes at a time in packed half precision. Codes j and j + 4 of a nibble word are 16 bits apart, where the halves want
// them; 64 + code is exact there, (64 + code) s - 96 s is too (6 bits of code - 32 times the 4 of s fit 11), and
// adding 1536 rounds to an integer, to nearest even, whose low byte is the result. A NaN scale gives -127, as there.
D3_INLINE i32x4 w6_group_i8_halves(uint32_t lo, uint32_t hi, uint32_t high, uint32_t scale_byte) {
  typedef _Float16 half2v __attribute__((ext_vector_type(2)));
  const _Float16 s = (_Float16)fp8x2_to_f32<false>(scale_byte).x;
  const half2v sv = {s, s}, c96 = sv * (_Float16)-96.0f;
  const half2v bottom = {(_Float16)-127.0f, (_Float16)-127.0f}, top = {(_Float16)127.0f, (_Float16)127.0f};
  const half2v magic = {(_Float16)1536.0f, (_Float16)1536.0f};
  i32x4 out;
#pragma unroll
  for (int d = 0; d < 2; d++) {
    const uint32_t word = d ? hi : lo;
    // the top bits of codes 8d .. 8d + 3 in the low half, of 8d + 4 .. 8d + 7 in the high one
    const uint32_t tops = __builtin_amdgcn_perm(0u, high, d ? 0x0C030C02u : 0x0C010C00u);
    uint32_t r[4];
#pragma unroll
    for (int j = 0; j < 4; j++) {
      const uint32_t nib = j == 0 ? word << 4 : word >> (4 * j - 4);
      const uint32_t bits = (nib & 0x00F000F0u) | (((tops << (8 - 2 * j)) & 0x03000300u) | 0x54005400u);  // 64 + code
      half2v t = __builtin_elementwise_fma(__builtin_bit_cast(half2v, bits), sv, c96);
      t = __builtin_elementwise_min(__builtin_elementwise_max(t, bottom), top);
      r[j] = __builtin_bit_cast(uint32_t, t + magic);
    }
    const uint32_t p01 = __builtin_amdgcn_perm(r[1], r[0], 0x06020400u);  // codes 0, 1, 4, 5
    const uint32_t p23 = __builtin_amdgcn_perm(r[3], r[2], 0x06020400u);  // codes 2, 3, 6, 7
    out[2 * d] = (int)__builtin_amdgcn_perm(p23, p01, 0x05040100u);
    out[2 * d + 1] = (int)__builtin_amdgcn_perm(p23, p01, 0x07060302u);
  }
  return out;
}

// A thread's share of a stage's codes: 64 columns of one weight row.
struct RawCodes {
  i32x4 low[2];
  i32x4 high;
  uint32_t scales;
};

// SWIGLU: the bank holds N / 2 gate rows, then N / 2 up rows. A workgroup takes 128 hidden units (in LDS 32 gate rows,
// then the same units' 32 up rows, per wave) and stores SiLU(gate) * up, [rows, N / 2], in place of both.
template <int KIND, bool SWIGLU>  // 0 int8, 4 / 6 codes
__global__ void __launch_bounds__(WT_THREADS, 2) wide_i8_kernel(WideArgs a) {
  constexpr bool CODES = KIND != 0;
  __shared__ __attribute__((aligned(1024))) uint8_t smem[2 * WI_STAGE];
  __shared__ __attribute__((aligned(16))) float factors[WT_N + 16 * WI_TILES];  // row (channel) scales, then the rows' plane scales
  __shared__ uint32_t qtab[KIND == 4 ? QTAB_WORDS : 1];
  const int N = a.N, K = a.K, stages = K / 128;
  const int RB = CODES ? K * KIND / 8 : K, G = K / 16;
  int pass, xb;
  wt_place(blockIdx.x, N / WT_N, pass, xb);
  if (pass >= a.count[0]) return;
  const int4 p4 = a.passes[pass];
  const int expert = __builtin_amdgcn_readfirstlane(p4.x), first = __builtin_amdgcn_readfirstlane(p4.y),
            rows = __builtin_amdgcn_readfirstlane(p4.z), tiles = (rows + 15) / 16;
  const int tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int q = lane >> 4, c = lane & 15, wn = w & 3, wm = w >> 2;
  const size_t n0 = (size_t)expert * N + (size_t)xb * (SWIGLU ? WT_N / 2 : WT_N);  // the workgroup's first bank row
  // the bank row, from n0, of the workgroup's row 32 * block + i, i < 32
  auto bank_row = [&](int block) { return SWIGLU ? 32 * (block >> 1) + (block & 1) * (N / 2) : 32 * block; };
  const uint32_t lds0 = lds_address(smem);

  // The rows' planes: 12 blocks of 8 rows x 3 planes, 36 copies of 1 KB dealt to the waves in turn (wave w: copies w,
  // w + 8, ...; copy i is block i % 12 of plane i / 12). A wave meets three different blocks.
  uint32_t xoff[3];
  {
    int p[3], own = first + min(max(tid - WT_N, 0), rows - 1);
#pragma unroll
    for (int i = 0; i < 3; i++) p[i] = first + min(8 * ((w + 8 * i) % 12) + (lane >> 3), rows - 1);
    if (a.order) {
#pragma unroll
      for (int i = 0; i < 3; i++) p[i] = (int)a.order[p[i]];
      own = (int)a.order[own];
#pragma unroll
      for (int i = 0; i < 3; i++) p[i] = pair_row(p[i], a.k_order, a.xrows);
      own = pair_row(own, a.k_order, a.xrows);
    }
#pragma unroll
    for (int i = 0; i < 3; i++)
      xoff[i] = (uint32_t)p[i] * (uint32_t)K + 16 * wt_slot(8 * ((w + 8 * i) % 12) + (lane >> 3), lane & 7);
    if (tid < WT_N) factors[tid] = (CODES ? a.c : (const float*)a.s)[n0 + bank_row(tid >> 5) + (tid & 31)];
    else if (tid < WT_N + 16 * WI_TILES) factors[tid] = a.xscale[own];
  }
  auto load_rows = [&](int stage, int buf, int i) __attribute__((always_inline)) {  // copy i < 5 of this wave
    const int n = w + 8 * i, b = n % 12, t = n / 12, mt = b >> 1;
    if (n < 36 && mt < tiles)
      dma16(lds0 + buf * WI_STAGE + WI_W_BYTES + (uint32_t)((mt * WI_PLANES + t) * 2048 + (b & 1) * 1024),
            a.xs + t * a.plane + 128 * stage, xoff[i % 3]);
  };
  // int8 weights: wave w copies rows 32 w .. 32 w + 31
  uint32_t woff[2];
#pragma unroll
  for (int i = 0; i < 2; i++) {
    const int r = 8 * i + (lane >> 3);
    woff[i] = (uint32_t)(r * K) + 16 * wt_slot(r, lane & 7);
  }
  const uint8_t* wwave = a.w + (n0 + bank_row(w)) * RB;
  auto load_weights = [&](int stage, int buf, int i) __attribute__((always_inline)) {  // copy i < 4 of this wave
    dma16(lds0 + buf * WI_STAGE + w * 4096 + 1024 * i, wwave + 128 * stage + (size_t)(i >> 1) * 16 * K, woff[i & 1]);
  };
  // codes: thread tid takes 64 columns (half tid & 1 of the stage) of row tid >> 1
  const int drow = tid >> 1, dhalf = tid & 1;
  const uint32_t doff = (uint32_t)((lane >> 1) * RB), dscale = (uint32_t)((lane >> 1) * G) + 4 * dhalf;
  const uint8_t* swave = (const uint8_t*)a.s + (n0 + bank_row(w)) * G;
  RawCodes raw;
  auto load_raw = [&](int stage) __attribute__((always_inline)) {
    raw.low[0] = *(const i32x4*)(wwave + 64 * stage + (doff + 32 * dhalf));
    raw.low[1] = *(const i32x4*)(wwave + 64 * stage + 16 + (doff + 32 * dhalf));
    if constexpr (KIND == 6) raw.high = *(const i32x4*)(wwave + K / 2 + 32 * stage + (doff + 16 * dhalf));
    raw.scales = *(const uint32_t*)(swave + 8 * stage + dscale);
  };
  auto decode = [&](int buf) __attribute__((always_inline)) {
    uint8_t* dst = smem + buf * WI_STAGE + drow * 128;
#pragma unroll
    for (int i = 0; i < 4; i++) {
      const uint32_t lo = (uint32_t)raw.low[i >> 1][2 * (i & 1)], hi = (uint32_t)raw.low[i >> 1][2 * (i & 1) + 1];
      const uint32_t sb = (raw.scales >> (8 * i)) & 0xFFu;
      i32x4 v;
      if constexpr (KIND == 4) v = w4_group_i8(lo, hi, *(const i32x4*)(qtab + 4 * sb));
      else v = w6_group_i8_halves(lo, hi, (uint32_t)raw.high[i], sb);
      *(i32x4*)(dst + 16 * wt_slot(drow, 4 * dhalf + i)) = v;
    }
  };
#pragma unroll
  for (int i = 0; i < 5; i++) load_rows(0, 0, i);
  if constexpr (CODES) {
    load_raw(0);
    if constexpr (KIND == 4) {
      build_qtab<true>(qtab, *(const f32x4*)(a.codebook + 4 * (tid & 3)));
      __syncthreads();
    }
    decode(0);
    load_raw(stages > 1 ? 1 : 0);
  } else {
#pragma unroll
    for (int i = 0; i < 4; i++) load_weights(0, 0, i);
  }

  // A wave's tiles: rows 16 (wm + 2 j) .., j < NT. Straight-line code per number of tiles, so that the next tile's
  // operands are on their way while one is multiplied.
  auto run = [&]<int NT>() __attribute__((always_inline)) {
    i32x4 acc[4][NT][WI_PLANES];
#pragma unroll
    for (int n = 0; n < 4; n++)
#pragma unroll
      for (int j = 0; j < NT; j++)
#pragma unroll
        for (int t = 0; t < WI_PLANES; t++) acc[n][j][t] = i32x4{0, 0, 0, 0};
    i32x4 wa[2][4], b[2][WI_PLANES];
    const int at0 = c * 128 + 16 * wt_slot(c, q), at1 = c * 128 + 16 * wt_slot(c, 4 + q);
    auto read_w = [&](int buf, int h) __attribute__((always_inline)) {
#pragma unroll
      for (int n = 0; n < 4; n++)
        wa[h][n] = *(const i32x4*)(smem + buf * WI_STAGE + (64 * wn + 16 * n) * 128 + (h ? at1 : at0));
    };
    auto read_x = [&](int buf, int h, int j, i32x4 (&v)[WI_PLANES]) __attribute__((always_inline)) {
#pragma unroll
      for (int t = 0; t < WI_PLANES; t++)
        v[t] = *(const i32x4*)(smem + buf * WI_STAGE + WI_W_BYTES + ((wm + 2 * j) * WI_PLANES + t) * 2048 + (h ? at1 : at0));
    };
    // Row tile J of half H of stage s: the next tile's operands are requested first, then the products; the next
    // stage's copies go out tile by tile (all at once they would hold the wave before its first product).
    auto block = [&]<int H, int J>(int s, bool more) __attribute__((always_inline)) {
      constexpr int I = H * NT + J, cur = I & 1;
      const int buf = s & 1;
      if constexpr (J + 1 < NT) {
        read_x(buf, H, J + 1, b[cur ^ 1]);
      } else if constexpr (H == 0) {
        read_w(buf, 1);
        read_x(buf, 1, 0, b[cur ^ 1]);
      }
      __builtin_amdgcn_sched_barrier(0);  // the reads first: left to itself the compiler issues each just before its use
      if (more) {
        constexpr int COPIES = CODES ? 5 : 9, PER = CODES || NT == 1 ? 5 : (COPIES + 2 * NT - 2) / (2 * NT - 1);
#pragma unroll
        for (int i = I * PER; i < (I + 1) * PER && i < COPIES; i++) {
          if (i < 5) load_rows(s + 1, buf ^ 1, i);
          else load_weights(s + 1, buf ^ 1, i - 5);
        }
      }
      // codes: the two waves of a SIMD decode the next stage's weights at different times, one's decoding beside the
      // other's products
      if constexpr (CODES && J == 0) {
        if (more && wm == H) {
          decode(buf ^ 1);
          if (s + 2 < stages) load_raw(s + 2);
        }
      }
#pragma unroll
      for (int t = 0; t < WI_PLANES; t++)
#pragma unroll
        for (int n = 0; n < 4; n++)
          acc[n][J][t] = __builtin_amdgcn_mfma_i32_16x16x64_i8(wa[H][n], b[cur][t], acc[n][J][t], 0, 0, 0);
      __builtin_amdgcn_sched_barrier(0);
    };
    dma_wait();
    __syncthreads();
    for (int s = 0; s < stages; s++) {
      const bool more = s + 1 < stages;
      read_w(s & 1, 0);
      read_x(s & 1, 0, 0, b[0]);
      block.template operator()<0, 0>(s, more);
      if constexpr (NT > 1) block.template operator()<0, 1>(s, more);
      if constexpr (NT > 2) block.template operator()<0, 2>(s, more);
      block.template operator()<1, 0>(s, more);
      if constexpr (NT > 1) block.template operator()<1, 1>(s, more);
      if constexpr (NT > 2) block.template operator()<1, 2>(s, more);
      dma_wait();
      __syncthreads();
    }

    // lane l holds weight rows 64 wn + 16 n + 4 q .. + 3 of the pass's row 16 mt + c
#pragma unroll
    for (int j = 0; j < NT; j++) {
      const int r = 16 * (wm + 2 * j) + c;
      if (r < rows) {
        const float sx = factors[WT_N + r];
        f32x4 v[4];
#pragma unroll
        for (int n = 0; n < 4; n++) {
          const f32x4 e = *(const f32x4*)(factors + 64 * wn + 16 * n + 4 * q);
#pragma unroll
          for (int i = 0; i < 4; i++)
            v[n][i] = e[i] * (sx * planes_sum(acc[n][j][0][i], acc[n][j][1][i], acc[n][j][2][i]));
        }
        if constexpr (SWIGLU) {
          float* o = a.out + (size_t)(first + r) * (N / 2) + xb * (WT_N / 2) + 32 * wn + 4 * q;
#pragma unroll
          for (int n = 0; n < 2; n++) {
            f32x4 h;
#pragma unroll
            for (int i = 0; i < 4; i++) h[i] = silu_up(v[n][i], v[n + 2][i]);
            *(f32x4*)(o + 16 * n) = h;
          }
        } else {
          float* o = a.out + (size_t)(first + r) * N + xb * WT_N + 64 * wn + 4 * q;
#pragma unroll
          for (int n = 0; n < 4; n++) *(f32x4*)(o + 16 * n) = v[n];
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

}  // namespace d3

using namespace d3;

extern "C" {

int d3_prompt_i8(int32_t kind, const void* planes, const float* scales, int64_t plane, const int64_t* order, int32_t k,
                 int32_t rows, const int32_t* passes, int64_t pass_ints, int32_t E, const void* w, const void* s,
                 const float* c, const float* codebook, float* out, int32_t N, int32_t K, int32_t swiglu, void* stream) {
  if (!planes || !scales || !passes || !w || !s || !out) return fail("d3_prompt_i8: null pointer");
  if (kind != 0 && kind != 4 && kind != 6) return fail("d3_prompt_i8: kind 0, 4 or 6");
  if (kind != 0 && !c) return fail("d3_prompt_i8: codes need channel scales");
  if (kind == 4 && !codebook) return fail("d3_prompt_i8: 4 bits need a codebook");
  if (N < WT_N || N % WT_N || K < 256 || K % 256 || K > 2048) return fail("d3_prompt_i8: N % 256 == 0, K % 256 == 0, K <= 2048");
  if (plane < K || plane % K || plane > (int64_t)UINT32_MAX - 4096) return fail("d3_prompt_i8: plane a multiple of K, under 2^32 bytes");
  if (rows < 1 || E < 1 || (order ? k < 1 : rows > plane / K))
    return fail("d3_prompt_i8: 1 <= rows (<= plane / K without order), k >= 1 with order");
  if ((((uintptr_t)planes | (uintptr_t)w) & 15) || (kind != 0 && ((uintptr_t)s & 3)))
    return fail("d3_prompt_i8: planes and weights at 16-byte, scale bytes at 4-byte alignment");
  if (pass_ints < d3_prompt_pass_ints(E, rows)) return fail("d3_prompt_i8: passes holds fewer than d3_prompt_pass_ints ints");
  WideArgs a;
  a.xs = (const int8_t*)planes;
  a.plane = plane;
  a.xscale = scales;
  a.order = order;
  a.k_order = k;
  a.xrows = (int)(plane / K);
  a.count = passes;
  a.passes = (const int4*)(passes + 4);
  a.w = (const uint8_t*)w;
  a.s = s;
  a.c = c;
  a.codebook = codebook;
  a.out = out;
  a.N = N;
  a.K = K;
  const int cap = rows / (16 * WI_TILES) + std::min(E, rows);
  const dim3 grid((unsigned)(wt_places(cap) * (N / WT_N)));
  const hipStream_t st = (hipStream_t)stream;
#define D3_WIDE(KD)                                                                                                  \
  if (swiglu) hipLaunchKernelGGL((wide_i8_kernel<KD, true>), grid, dim3(WT_THREADS), 0, st, a);                      \
  else hipLaunchKernelGGL((wide_i8_kernel<KD, false>), grid, dim3(WT_THREADS), 0, st, a);                            \
  break
  switch (kind) {
    case 0: D3_WIDE(0);
    case 4: D3_WIDE(4);
    default: D3_WIDE(6);
  }
#undef D3_WIDE
  const hipError_t e = hipGetLastError();
  return e == hipSuccess ? 0 : hip_fail(e, "d3_prompt_i8");
}

}  // extern "C"
