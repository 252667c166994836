// The grouped products of a long prompt on A8 banks. moe_prefill.hip's grouped_kernel walks an expert's rows 16 at a
// time past 32 weight rows held in registers, and reads every row's activations from L2 once per 32 weight rows: 48
// times over for the first bank. That suits experts with a few rows; with hundreds, this kernel's tiles read both
// operands from L2 a fourth to an eighth as often: 256 x 256 (int8), 256 weight rows x 128 (FP8) or 128 x 128 (W4,
// W6), a wave's 64 weight rows from LDS, two waves per SIMD.
// Measured, 4096 rows, top-8 of 128 experts (FFN 768), first / second bank's products in a kernel trace: int8 511 /
// 262 us before, 182 / 140 here, FP8 234 / 174, W4 230 / 161, W6 261 / 178; the layer untraced: int8 874 / 400, FP8
// 879 / 485, W4 807 / 459, W6 882 / 513 (8192 rows, Zipf routing: int8 1703 / 706). The banks' and results' bytes take
// about 105 us of each int8 product at the rate a copy reaches and the products 100 and 50: they overlap within a
// workgroup, but its first loads and its stores do not.
// W4 and W6 as one workgroup of 256 x 128 per CU took 512 and 576 us a layer there, as 128 x 256 522 and 575; two of
// 128 x 128 read more from L2 and cover each other's first loads, barriers and stores. (256 x 256 with the columns'
// groups added in one run, which needs one set of accumulators, took 437 and 489, and 229 where two workgroups take
// 188 for 1024 rows with Zipf routing.)
#include "a8_wide.hpp"
#include "formats.hpp"

#include <type_traits>

namespace d3 {
namespace {

// acc[n] += A[n] . B, e4m3, four 16 x 16 x 128 products. One statement, as mfma_f8_chain (formats.hpp): the operands
// keep their registers until the products have read them, and the wait states before and after cover the
// instruction's hazards, which the compiler does not see inside.
D3_INLINE void mfma_f8_4(f32x4 (&acc)[4], const i32x8 (&A)[4], i32x8 B) {
  const int one = 127;  // E8M0 block scale 2^0
  asm volatile(
      "s_nop 4\n"
      "v_mfma_scale_f32_16x16x128_f8f6f4 %0, %4, %8, %0, %9, %9 op_sel_hi:[0,0,0]\n"
      "v_mfma_scale_f32_16x16x128_f8f6f4 %1, %5, %8, %1, %9, %9 op_sel_hi:[0,0,0]\n"
      "v_mfma_scale_f32_16x16x128_f8f6f4 %2, %6, %8, %2, %9, %9 op_sel_hi:[0,0,0]\n"
      "v_mfma_scale_f32_16x16x128_f8f6f4 %3, %7, %8, %3, %9, %9 op_sel_hi:[0,0,0]\n"
      "s_nop 7\n s_nop 7\n s_nop 7\n"
      : "+v"(acc[0]), "+v"(acc[1]), "+v"(acc[2]), "+v"(acc[3])
      : "v"(A[0]), "v"(A[1]), "v"(A[2]), "v"(A[3]), "v"(B), "v"(one));
}

// s + a b, the product rounded by itself (grouped_kernel's waves exchange such products)
D3_INLINE float add_product(float s, float a, float b) {
#pragma clang fp contract(off)
  const float p = a * b;
  return s + p;
}

// gate_up (DOWN false): a workgroup's columns are half as many hidden units, in LDS 32 gate rows and the same units' 32 up
// rows per 64.
template <int F, bool DOWN>
__global__ void __launch_bounds__(2 * a8_wide_cols(F), 2) a8_wide_kernel(A8WideArgs a) {
  constexpr int TILES = a8_wide_tiles(F), AW_ROWS = 16 * TILES, AW_N = a8_wide_cols(F);
  constexpr int AW_W_BYTES = AW_N * 128, AW_STAGE = AW_W_BYTES + AW_ROWS * 128;
  constexpr int WN = AW_N / 64, WAVES = 2 * WN;  // WN over the weight rows (64 each), two over the pass's tiles (in turn)
  constexpr int COPIES = 2 * TILES / WAVES;      // of 8 rows, per wave
  constexpr bool GROUPS = group_scaled(F);  // W4, W6: a scale per 128 columns, and codes to unpack
  constexpr int SRB = step_row_bytes(F);    // a stage's bytes of a weight row
  __shared__ __attribute__((aligned(1024))) uint8_t smem[2 * AW_STAGE];
  __shared__ __attribute__((aligned(16))) float wscale[GROUPS ? 2 : 1][AW_N];  // row scales, or a stage's group scales
  __shared__ float xscale[AW_ROWS];
  __shared__ int out_row[AW_ROWS];
  const int N = a.N, K = a.K, stages = K / 128, RB = stages * SRB;
  int pass, xb;
  wt_place(blockIdx.x, N / AW_N, pass, xb);
  if (pass >= a.count[0]) return;
  const int4 p4 = a.passes[pass];
  const int expert = __builtin_amdgcn_readfirstlane(p4.x), first = __builtin_amdgcn_readfirstlane(p4.y),
            rows = __builtin_amdgcn_readfirstlane(p4.z), tiles = (rows + 15) / 16;
  const int tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int q = lane >> 4, c = lane & 15, wn = w % WN, wm = w / WN;
  const size_t n0 = (size_t)expert * N + (size_t)xb * (DOWN ? AW_N : AW_N / 2);  // the workgroup's first bank row
  // the bank row, from n0, of the workgroup's row 32 * block + i, i < 32
  auto bank_row = [&](int block) { return DOWN ? 32 * block : 32 * (block >> 1) + (block & 1) * (N / 2); };
  const uint32_t lds0 = lds_address(smem);

  // the pass's rows: copies of 8 rows, wave w takes copies w, w + WAVES, ...
  uint32_t xoff[COPIES];
  {
    int p[COPIES];
#pragma unroll
    for (int i = 0; i < COPIES; i++) p[i] = first + min(8 * (w + WAVES * i) + (lane >> 3), rows - 1);
    if constexpr (!DOWN) {
#pragma unroll
      for (int i = 0; i < COPIES; i++) p[i] = a.perm[p[i]];
#pragma unroll
      for (int i = 0; i < COPIES; i++) p[i] /= a.k;
    }
#pragma unroll
    for (int i = 0; i < COPIES; i++)
      xoff[i] = (uint32_t)p[i] * (uint32_t)K + 16 * wt_slot(8 * (w + WAVES * i) + (lane >> 3), lane & 7);
    if (tid < AW_ROWS) {
      const int sp = first + min(tid, rows - 1), pair = a.perm[sp];
      out_row[tid] = pair;
      xscale[tid] = a.act_scale[DOWN ? sp : pair / a.k];
    }
    if (!GROUPS && tid >= AW_N) {
      const int r = tid - AW_N;
      wscale[0][r] = bf16_to_f32(a.s[n0 + bank_row(r >> 5) + (r & 31)]);
    }
  }
  auto load_rows = [&](int stage, int buf) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < COPIES; i++)
      if ((w + WAVES * i) >> 1 < tiles)
        dma16(lds0 + buf * AW_STAGE + AW_W_BYTES + (uint32_t)(w + WAVES * i) * 1024, a.act + 128 * stage, xoff[i]);
  };
  const uint8_t* wwave = a.w + (n0 + bank_row(w)) * RB;
  // bytes (int8, e4m3): wave w copies rows 32 w .. 32 w + 31
  uint32_t woff[2];
#pragma unroll
  for (int i = 0; i < 2; i++) {
    const int r = 8 * i + (lane >> 3);
    woff[i] = (uint32_t)(r * RB) + 16 * wt_slot(r, lane & 7);
  }
  auto load_weights = [&](int stage, int buf) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < 4; i++)
      dma16(lds0 + buf * AW_STAGE + w * 4096 + 1024 * i, wwave + 128 * stage + (size_t)(i >> 1) * 16 * RB, woff[i & 1]);
  };
  // codes: thread tid takes 64 columns (half tid & 1 of the stage) of row tid >> 1
  constexpr int RAW = GROUPS ? SRB / 32 : 1;  // 16-byte words of that
  const int drow = tid >> 1, dhalf = tid & 1;
  const uint32_t doff = (uint32_t)((lane >> 1) * RB + (SRB / 2) * dhalf);
  i32x4 raw[RAW];
  uint32_t raw_scale = 0;
  auto load_raw = [&](int stage) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < RAW; i++) raw[i] = *(const i32x4*)(wwave + SRB * stage + 16 * i + doff);
    if (tid < AW_N) raw_scale = a.s[(n0 + bank_row(tid >> 5) + (tid & 31)) * stages + stage];
  };
  auto unpack = [&](int buf) __attribute__((always_inline)) {
    uint8_t* dst = smem + buf * AW_STAGE + drow * 128;
#pragma unroll
    for (int i = 0; i < 4; i++) {
      i32x4 v;
      if constexpr (F == FMT_W4) {
        uint32_t e0, o0, e1, o1;
        unpack_w4_word((uint32_t)raw[i >> 1][2 * (i & 1)], e0, o0);
        unpack_w4_word((uint32_t)raw[i >> 1][2 * (i & 1) + 1], e1, o1);
        v = i32x4{(int)e0, (int)o0, (int)e1, (int)o1};
      } else {
        const int d = 3 * i;
        v = unpack_w6_unit((uint32_t)raw[(d / 4) % RAW][d & 3], (uint32_t)raw[((d + 1) / 4) % RAW][(d + 1) & 3],
                           (uint32_t)raw[((d + 2) / 4) % RAW][(d + 2) & 3]);
      }
      *(i32x4*)(dst + 16 * wt_slot(drow, 4 * dhalf + i)) = v;
    }
    // the unpacked codes carry a factor 2^unpack_shift, taken out of the group scale (exactly)
    if (tid < AW_N) wscale[GROUPS ? buf : 0][tid] = bf16_to_f32(raw_scale) * (1.0f / (1 << unpack_shift(F)));
  };
  load_rows(0, 0);
  if constexpr (GROUPS) {
    load_raw(0);
    unpack(0);
    load_raw(min(1, stages - 1));
  } else {
    load_weights(0, 0);
  }

  // A wave's tiles: rows 16 (wm + 2 j) .., j < NT (tiles past the pass's run on what lies there and store nothing)
  auto run = [&]<int NT>() __attribute__((always_inline)) {
    typedef typename std::conditional<F == FMT_I8, i32x4, f32x4>::type Acc;
    Acc acc[NT][4];
#pragma unroll
    for (int j = 0; j < NT; j++)
#pragma unroll
      for (int n = 0; n < 4; n++) acc[j][n] = Acc{0, 0, 0, 0};
    // float32 sums: those of the K slices before this one, and the slices' length (grouped_kernel's: 4 slices of the
    // first bank's K, 2 of the second's)
    f32x4 sum[F == FMT_I8 ? 1 : NT][4];
    const int slice = stages / (DOWN ? 2 : 4);
    int left = slice;
    if constexpr (F != FMT_I8) {
#pragma unroll
      for (int j = 0; j < NT; j++)
#pragma unroll
        for (int n = 0; n < 4; n++) sum[j][n] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    }
    i32x4 wa[4][2], b[2][2];
    // a lane's columns of a stage: pieces 2 q and 2 q + 1, the 32 that grouped_kernel's lanes take (FP8's products add
    // their columns in lane order)
    const int at0 = c * 128 + 16 * wt_slot(c, 2 * q), at1 = c * 128 + 16 * wt_slot(c, 2 * q + 1);
    auto read_x = [&](int buf, int j, i32x4 (&v)[2]) __attribute__((always_inline)) {
      const uint8_t* src = smem + buf * AW_STAGE + AW_W_BYTES + (wm + 2 * j) * 2048;
      v[0] = *(const i32x4*)(src + at0);
      v[1] = *(const i32x4*)(src + at1);
    };
    dma_wait();
    __syncthreads();
    for (int s = 0; s < stages; s++) {
      const int buf = s & 1;
      const bool more = s + 1 < stages;
#pragma unroll
      for (int n = 0; n < 4; n++) {
        const uint8_t* src = smem + buf * AW_STAGE + (64 * wn + 16 * n) * 128;
        wa[n][0] = *(const i32x4*)(src + at0);
        wa[n][1] = *(const i32x4*)(src + at1);
      }
      read_x(buf, 0, b[0]);
      f32x4 g[4];
      if constexpr (GROUPS) {
#pragma unroll
        for (int n = 0; n < 4; n++) g[n] = *(const f32x4*)(wscale[buf] + 64 * wn + 16 * n + 4 * q);
      }
      if (more) {
        if constexpr (GROUPS) unpack(buf ^ 1);
        load_rows(s + 1, buf ^ 1);
        if constexpr (GROUPS) load_raw(min(s + 2, stages - 1));
        else load_weights(s + 1, buf ^ 1);
      }
#pragma unroll
      for (int j = 0; j < NT; j++) {
        if (j + 1 < NT) read_x(buf, j + 1, b[(j + 1) & 1]);
        __builtin_amdgcn_sched_barrier(0);  // the reads first
        if constexpr (F == FMT_I8) {
#pragma unroll
          for (int h = 0; h < 2; h++)
#pragma unroll
            for (int n = 0; n < 4; n++) acc[j][n] = mfma_i8(wa[n][h], b[j & 1][h], acc[j][n]);
        } else if constexpr (F == FMT_F8) {
          i32x8 A[4];
#pragma unroll
          for (int n = 0; n < 4; n++) A[n] = f8_operand(wa[n][0], wa[n][1]);
          mfma_f8_4(acc[j], A, f8_operand(b[j & 1][0], b[j & 1][1]));
        } else {
          i32x4 d[4];
#pragma unroll
          for (int n = 0; n < 4; n++) d[n] = mfma_i8(wa[n][0], b[j & 1][0], i32x4{0, 0, 0, 0});
#pragma unroll
          for (int n = 0; n < 4; n++) d[n] = mfma_i8(wa[n][1], b[j & 1][1], d[n]);
#pragma unroll
          for (int n = 0; n < 4; n++)
#pragma unroll
            for (int i = 0; i < 4; i++) acc[j][n][i] = fmaf((float)d[n][i], g[n][i], acc[j][n][i]);
        }
      }
      if constexpr (F != FMT_I8) {
        if (--left == 0) {  // the slice's sums (FP8: scaled) onto the earlier ones'
          left = slice;
#pragma unroll
          for (int n = 0; n < 4; n++) {
            f32x4 rs;
            if constexpr (F == FMT_F8) rs = *(const f32x4*)(wscale[0] + 64 * wn + 16 * n + 4 * q);
#pragma unroll
            for (int j = 0; j < NT; j++) {
#pragma unroll
              for (int i = 0; i < 4; i++) {
                if constexpr (F == FMT_F8) sum[j][n][i] = add_product(sum[j][n][i], acc[j][n][i], rs[i]);
                else sum[j][n][i] += acc[j][n][i];
              }
              acc[j][n] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
            }
          }
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
        const float xs = xscale[r];
        f32x4 v[4];
#pragma unroll
        for (int n = 0; n < 4; n++) {
          f32x4 rs;
          if constexpr (F == FMT_I8) rs = *(const f32x4*)(wscale[0] + 64 * wn + 16 * n + 4 * q);
#pragma unroll
          for (int i = 0; i < 4; i++) {
            if constexpr (F == FMT_I8) v[n][i] = (float)acc[j][n][i] * rs[i] * xs;
            else v[n][i] = sum[j][n][i] * xs;
          }
        }
        if constexpr (DOWN) {
          float* o = a.out + (size_t)out_row[r] * N + xb * AW_N + 64 * wn + 4 * q;
#pragma unroll
          for (int n = 0; n < 4; n++) *(f32x4*)(o + 16 * n) = v[n];
        } else {
          float* o = a.out + (size_t)(first + r) * (N / 2) + xb * (AW_N / 2) + 32 * wn + 4 * q;
#pragma unroll
          for (int n = 0; n < 2; n++) {
            f32x4 h;
#pragma unroll
            for (int i = 0; i < 4; i++) h[i] = v[n][i] / (1.0f + __expf(-v[n][i])) * v[n + 2][i];
            *(f32x4*)(o + 16 * n) = h;
          }
        }
      }
    }
  };
  const int pairs = (tiles - wm + 3) / 4;  // of this wave's tiles
  if constexpr (TILES > 8) {
    if (pairs == 4) return run.template operator()<8>();
    if (pairs == 3) return run.template operator()<6>();
  }
  if (pairs >= 2) run.template operator()<4>();
  else run.template operator()<2>();
}

}  // namespace

void launch_a8_wide(int format, bool down, const A8WideArgs& a, int cap, hipStream_t s) {
  const dim3 grid((unsigned)(wt_places(cap) * (a.N / a8_wide_cols(format)))), block(2 * a8_wide_cols(format));
#define D3_AW(F)                                                                                    \
  if (down) hipLaunchKernelGGL((a8_wide_kernel<F, true>), grid, block, 0, s, a);                     \
  else hipLaunchKernelGGL((a8_wide_kernel<F, false>), grid, block, 0, s, a);                        \
  break
  switch (format) {
    case FMT_I8: D3_AW(FMT_I8);
    case FMT_W4: D3_AW(FMT_W4);
    case FMT_W6: D3_AW(FMT_W6);
    default: D3_AW(FMT_F8);
  }
#undef D3_AW
}

}  // namespace d3
