// The MFMA layer of the 64 -> 128 -> 1 trajectory kernel: both contractions of a 16-row tile on
// v_mfma_f32_16x16x32_bf16 with every FP32 operand split into three bf16 parts, the pointwise stage between
// them, the tile loop and the wave's partial sums.  In a header of its own so that the tile-ceiling probe
// (tile_ceiling.hip) times exactly the code the kernel runs.
#pragma once

#include <hip/hip_runtime.h>

#include "bnn_device.h"
#include "bnn_kernel_common.h"
#include "bnn_split_bf16.h"

namespace bnn {

// ================================================================================================
// Lane l = 16 q + n.  Per 16-row tile:
//   GEMM1  A = X tile [16 rows x 32 k]    lane (n, q) holds row n, k = 32 kc + 8 q + i (i < 8)
//          B = W1 [32 k x 16 c]           three parts in LDS, one 16-byte read per lane, part, kc and t
//          C = pre-activation             lane (n, q) holds rows 4 q + j, c = 16 t + n (bias as C init)
//   GEMM2  A = u^T = C registers as they are, split: two parts of rows 4 q + j fill the eight k slots
//          B = g X [16 rows x 16 f]       lane (n, q) holds rows 4 q + j, features 32 v + 2 n + u, split
//          C = dW1^T [16 c x 16 f]        lane (n, q) holds c = 16 t + 4 q + j', f = 32 v + 2 n + u
//
// Why split: v_mfma_f32_16x16x4_f32 runs at 64 flop per cycle and SIMD and shares its pipe with the vector
// instructions; the bf16 form runs at 1024 on a pipe of its own.  x = h + m + l with three bf16 parts is exact
// for a 24-bit significand, and the six products hh, hm, mh, hl, lh, mm leave out ml, lm and ll, of random sign and
// 2^-27 of a product each on average (2^-24 at most): less than the FP32 rounding of one addition, of which GEMM1 has
// 12 per 64 products (six of the parts per 32) instead of 16, GEMM2 three per tile instead of four.  So the contraction costs 6/16 of the FP32 time, off the vector pipe, at
// FP32 precision (measured against 64 bits: as close or closer).  A tile took 4.46 us per SIMD, now 2.5; what limits
// it is power (the shader clock drops from 2.39 to 2.1 GHz).
// GEMM2 has only 16 rows to contract per tile and 32 k slots per instruction: two products share an
// instruction, [m | h] x [h | m], [h | l] x [l | h] and [h | m] x [h | m].
// ================================================================================================
template <int D0, int D1>
struct MfmaWideLayer {
  static_assert(D0 % 32 == 0 && D1 % 16 == 0, "tiles must divide the layer sizes");
  static constexpr int KC = D0 / 32;  // k chunks of GEMM1
  static constexpr int NT = D1 / 16;
  static constexpr int D1_ = D1;
  static constexpr int FV = D0 / 32;
  static constexpr int FT = 2 * FV;
  static constexpr int oB1 = D0 * D1, oW2 = oB1 + D1, oB2 = oW2 + D1, P = oB2 + 1;
  static constexpr int P_AL = (P + 3) / 4 * 4;
  // W1 split: part-major, then [kc][t][lane][8 bf16], so that a wave's read of a fragment is linear
  static constexpr int PLANE = D0 * D1;
  static constexpr int PLANES_BYTES = 3 * PLANE * 2;
  static constexpr float kExp2Scale = -2.88539008177792681472f;  // -2 / ln 2, kernel_helpers.h:37

  f4 dacc[NT][FT];
  float dw2acc[NT];
  float db1acc[NT];
  float db2acc;
  double dl;
  // per step (prepare_step): every lane's part of the layer-2 sum starts from its own share of the
  // constant (sum of w2 - b2) sr2; what the roundings of the 16 shares leave over, and the target
  // times sr2, are added to the finished row sum.  sr2 is the power of two next to 1 / scale, the factor
  // (1 / scale) / sr2 is applied to the finished sum
  float y_0, rho, sr2v, ratio, w2_scale;  // w2_scale = -2 sr2

  // offset of parameter (k, c) of W1 in a part
  static __device__ __forceinline__ int plane_offset(int k, int c) {
    return (((k >> 5) * NT + (c >> 4)) * 64 + ((k >> 3) & 3) * 16 + (c & 15)) * 8 + (k & 7);
  }
  // W1 scaled by -2 / ln 2 (GEMM1 then yields the exp2 argument directly) and split: the eight weights
  // (8 o + i, c), which lie one behind the other in a part
  static __device__ __forceinline__ void store_split8(__bf16* planes, int o, int c, const float (&w)[8]) {
    bf8 h, m, l;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      __bf16 ph, pm, pl;
      split_scaled(w[i], kExp2Scale, ph, pm, pl);
      h[i] = ph;
      m[i] = pm;
      l[i] = pl;
    }
    __bf16* dst = planes + plane_offset(8 * o, c);
    *reinterpret_cast<bf8*>(dst) = h;
    *reinterpret_cast<bf8*>(dst + PLANE) = m;
    *reinterpret_cast<bf8*>(dst + 2 * PLANE) = l;
  }

  // rows of X as the two contractions take them, and the target of row 4 q + (n >> 2): lane n sits in bank
  // n >> 2, where that row's sum lands
  struct RowsA {
    f4 x[KC][2];
  };
  struct RowsB {
    f2 x[4][FV];
    float y1;
  };

  __device__ __forceinline__ void zero_acc() {
#pragma unroll
    for (int t = 0; t < NT; ++t) {
#pragma unroll
      for (int ft = 0; ft < FT; ++ft) dacc[t][ft] = f4{0.f, 0.f, 0.f, 0.f};
      dw2acc[t] = 0.0f;
      db1acc[t] = 0.0f;
    }
    db2acc = 0.0f;
    dl = 0.0;
  }

  // The pointwise stage works with s = 1 / (1 + 2^t) = (1 + tanh x) / 2 and never forms h = 2 s - 1:
  //   yhat = sum w2 h + b2 = 2 sum w2 s - (sum w2 - b2)        (the constant: once per step, in double)
  //   dw2  = sum g h       = 2 sum g s - sum g                  (add_partials)
  //   1 - h^2 = 4 (s - s^2)                                     (the 4 goes into add_partials)
  // Scaling by a power of two keeps every product of the layer-2 sum exact.
  __device__ __forceinline__ void prepare_step(const float* s_w, const ModelConsts& mc) {
    const int lane = opaque_tid() & 63, n = lane & 15;
    const uint32_t sr2_bits = (__builtin_bit_cast(uint32_t, mc.scale_recp) + 0x00400000u) & 0x7F800000u;
    const float sr2 = __builtin_bit_cast(float, sr2_bits);
    ratio = mc.scale_recp * __builtin_bit_cast(float, 0x7F000000u - sr2_bits);
    // the share of lane n: its hidden units 16 t + n [and b2 in lane 0]; a large constant in one lane
    // would set the rounding grid of that lane's whole sum, and where hidden units saturate the terms
    // take few distinct values, so roundings would repeat from row to row instead of averaging out
    double share = 0.0;
#pragma unroll
    for (int t = 0; t < NT; ++t) share += (double)s_w[oW2 + 16 * t + n];
    if (n == 0) share -= (double)s_w[oB2];
    share *= (double)sr2;
    y_0 = (float)share;
    const double rest = row16_allreduce_d(share - (double)y_0);
    rho = __builtin_bit_cast(float, __builtin_amdgcn_readfirstlane(__builtin_bit_cast(int, (float)rest)));
    sr2v = sr2;
    w2_scale = -2.0f * sr2;
  }

  // FULL: sixteen rows, 16-byte aligned; a wave-uniform base and a per-lane 32-bit offset that stays the same, so
  // that no vector instruction is spent on addresses.  Otherwise any alignment, and rows past the end read as the
  // last row (their gradient is masked to zero).
  template <bool FULL>
  static __device__ __forceinline__ void load_a(RowsA& ra, const StepCtx& cx, int row0, int n, int q) {
    if (FULL) {
      const char* base = reinterpret_cast<const char*>(cx.X + (size_t)row0 * D0);
      const unsigned off = (unsigned)(n * D0 + 8 * q) * 4;
#pragma unroll
      for (int kc = 0; kc < KC; ++kc) {
#pragma unroll
        for (int i = 0; i < 2; ++i) ra.x[kc][i] = *reinterpret_cast<const f4*>(base + off + 128 * kc + 16 * i);
      }
    } else {
      const float* r = cx.X + (size_t)min(row0 + n, cx.n - 1) * D0 + 8 * q;
#pragma unroll
      for (int kc = 0; kc < KC; ++kc) {
#pragma unroll
        for (int i = 0; i < 2; ++i) {
          const float* e = r + 32 * kc + 4 * i;
          ra.x[kc][i] = f4{e[0], e[1], e[2], e[3]};
        }
      }
    }
  }
  template <bool FULL>
  static __device__ __forceinline__ void load_b(RowsB& rb, const StepCtx& cx, int row0, int n, int q) {
    if (FULL) {
      const char* base = reinterpret_cast<const char*>(cx.X + (size_t)row0 * D0);
      const unsigned off = (unsigned)(4 * q * D0 + 2 * n) * 4;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
#pragma unroll
        for (int v = 0; v < FV; ++v) rb.x[j][v] = *reinterpret_cast<const f2*>(base + off + 4 * D0 * j + 128 * v);
      }
      const char* by = reinterpret_cast<const char*>(cx.y + row0);
      rb.y1 = *reinterpret_cast<const float*>(by + (unsigned)(4 * q + (n >> 2)) * 4);
    } else {
      const int last = cx.n - 1;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const float* r = cx.X + (size_t)min(row0 + 4 * q + j, last) * D0 + 2 * n;
#pragma unroll
        for (int v = 0; v < FV; ++v) rb.x[j][v] = f2{r[32 * v], r[32 * v + 1]};
      }
      rb.y1 = cx.y[min(row0 + 4 * q + (n >> 2), last)];
    }
  }

  // GEMM1 of a tile in FP32, the rows read again from memory (rows past the end: the last row); scaled afterwards, since
  // -2 / ln 2 times a large finite weight may be infinite
  static __device__ __forceinline__ void gemm1_fp32(const float* s_w, const StepCtx& cx, int row0, int n, int q,
                                                    f4 (&acc)[NT]) {
    const float* row = cx.X + (size_t)min(row0 + n, cx.n - 1) * D0;
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      const float b = s_w[oB1 + 16 * t + n];
      acc[t] = f4{b, b, b, b};
    }
#pragma unroll 1
    for (int k = q; k < D0; k += 4) {
      const float x = row[k];
      const float* w = s_w + k * D1 + n;
#pragma unroll
      for (int t = 0; t < NT; ++t) acc[t] = mfma_f32(x, w[16 * t], acc[t]);
    }
#pragma unroll
    for (int t = 0; t < NT; ++t) acc[t] *= kExp2Scale;
  }

  // GEMM1 + activation + loss gradient + GEMM2 of one tile; `mid` runs before the pointwise stage and `late` in
  // the middle of GEMM2 (the tile loop issues loads there, as registers become free).  PARTS is for
  // the tile-ceiling probe, which times the halves of the instruction mix alone: 1 = the matrix instructions,
  // their operand fetch from LDS and the splits, 2 = the pointwise stage, 3 = the whole tile (what the kernel runs).
  // FP32: where a row sum is NaN, GEMM1 in FP32.
  template <int LIK, bool LAST, bool FULL, int PARTS = 3, bool FP32 = false, class Mid, class Late>
  __device__ __forceinline__ void compute_tile(const RowsA& ra, RowsB& rb, const float* s_w, const __bf16* planes,
                                               const StepCtx& cx, const ModelConsts& mc, int row0, int n, int q,
                                               Mid mid, Late late) {
    // what is read from LDS here does not change from tile to tile; an offset the compiler cannot see through
    // keeps it from holding all of it in registers
    int zero = 0;
    asm volatile("" : "+s"(zero));
    s_w += zero;
    planes += zero;
    f4 acc[NT];
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      const float b = s_w[oB1 + 16 * t + n] * kExp2Scale;
      acc[t] = f4{b, b, b, b};
    }
    if (PARTS & 1) {
      // fragments of W1 are read one hidden tile ahead; the scheduling fences keep the compiler from reading
      // more of them early than there are registers for
      const __bf16* frag = planes + 8 * (16 * q + n);
      bf8 bw[2][3];
      auto read = [&](int i) {
#pragma unroll
        for (int part = 0; part < 3; ++part)
          bw[i & 1][part] = *reinterpret_cast<const bf8*>(frag + i * 512 + part * PLANE);
      };
      read(0);
      bf8 ah, am, al;
#pragma unroll
      for (int i = 0; i < KC * NT; ++i) {
        const int kc = i / NT, t = i % NT;
        if (t == 0) split8<true>(ra.x[kc][0], ra.x[kc][1], ah, am, al);
        if (i + 1 < KC * NT) read(i + 1);
        const bf8 bh = bw[i & 1][0], bm = bw[i & 1][1], bl = bw[i & 1][2];
        acc[t] = mfma_bf16(al, bh, acc[t]);
        acc[t] = mfma_bf16(ah, bl, acc[t]);
        acc[t] = mfma_bf16(am, bm, acc[t]);
        acc[t] = mfma_bf16(am, bh, acc[t]);
        acc[t] = mfma_bf16(ah, bm, acc[t]);
        acc[t] = mfma_bf16(ah, bh, acc[t]);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
    if (PARTS == 2) {  // probe only: unknown pre-activations
#pragma unroll
      for (int t = 0; t < NT; ++t) asm volatile("" : "+v"(acc[t]));
    }
    mid();
    f2 gx[4][FV];
    if (PARTS & 2) {
      // s = 1 / (1 + 2^t) (kernel_helpers.h:34-42 without the small-|x| identity branch, see prepare_step)
      float rz;
      auto row_sums = [&] {
        float yh[4] = {y_0, y_0, y_0, y_0};
#pragma unroll
        for (int t = 0; t < NT; ++t) {
          const float w2y = s_w[oW2 + 16 * t + n] * w2_scale;
#pragma unroll
          for (int j = 0; j < 4; ++j) {
            const float e = __builtin_amdgcn_exp2f(acc[t][j]);
            const float sg = __builtin_amdgcn_rcpf(1.0f + e);
            acc[t][j] = sg;
            yh[j] = __builtin_fmaf(w2y, sg, yh[j]);
          }
        }
        rz = row16_reduce4(yh[0], yh[1], yh[2], yh[3]) + __builtin_fmaf(rb.y1, sr2v, rho);
      };
      row_sums();
      if constexpr (FP32) {
        if (__builtin_amdgcn_ballot_w64(__builtin_isnan(rz)) != 0) {
          gemm1_fp32(s_w, cx, row0, n, q, acc);
          row_sums();
        }
      }
      // scaled residual (y - yhat - b2) / scale of the four rows 4 q + j (mcmc_step_ffma.h:293), in bank
      // j of one register; the loss gradient is computed on that one register
      const float dz = rz * ratio;
      float gz;
      if (LIK == 0) gz = dz * mc.g_scale * __builtin_amdgcn_rcpf(__builtin_fmaf(dz, dz, mc.df));
      else gz = dz * mc.scale_recp;
      float g[4] = {row16_bcast<0>(gz), row16_bcast<1>(gz), row16_bcast<2>(gz), row16_bcast<3>(gz)};
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const bool valid = FULL || (row0 + 4 * q + j < cx.n);
        g[j] = valid ? g[j] : 0.0f;  // mcmc_step_ffma.h:301
        db2acc += g[j];
      }
      if (LAST) {
        // every lane holds the residual of its bank's row: the four rows of a lane group at once, stored and summed
        // by the first lane of each bank
        const int row = row0 + 4 * q + (n >> 2);
        const float lv = lik_value<LIK>(mc, dz);
        if ((n & 3) == 0 && (FULL || row < cx.n)) {
          const float prev = cx.ell_prev ? cx.ell_prev[row] : 0.0f;
          if (cx.ell_new) cx.ell_new[row] = lv;
          dl += (double)(lv - prev);
        }
      }
      // GEMM2 operands: u = s - s^2 stays where it is (A), g goes into the rows of x (B); the factors
      // 4 w2[c] of delta are applied once per step to the sums
#pragma unroll
      for (int t = 0; t < NT; ++t) {
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const float sg = acc[t][j];
          dw2acc[t] = __builtin_fmaf(g[j], sg, dw2acc[t]);
          const float u = __builtin_fmaf(-sg, sg, sg);
          acc[t][j] = u;
          db1acc[t] = __builtin_fmaf(u, g[j], db1acc[t]);
        }
      }
#pragma unroll
      for (int j = 0; j < 4; ++j) {
#pragma unroll
        for (int v = 0; v < FV; ++v) gx[j][v] = rb.x[j][v] * g[j];
      }
    } else {  // probe only: the matrix instructions on the raw operands
#pragma unroll
      for (int j = 0; j < 4; ++j) {
#pragma unroll
        for (int v = 0; v < FV; ++v) gx[j][v] = rb.x[j][v];
      }
    }
    if (PARTS & 1) {
      bf8 b_hm[FT], b_lh[FT];
#pragma unroll
      for (int ft = 0; ft < FT; ++ft) {
        bf4 h, m, l;
        split4<true>(f4{gx[0][ft >> 1][ft & 1], gx[1][ft >> 1][ft & 1], gx[2][ft >> 1][ft & 1], gx[3][ft >> 1][ft & 1]}, h,
               m, l);
        b_hm[ft] = join(h, m);
        b_lh[ft] = join(l, h);
      }
#pragma unroll
      for (int t = 0; t < NT; ++t) {
        if (t == NT / 2) late();
        bf4 h, m, l;
        split4<true>(acc[t], h, m, l);
        const bf8 a_mh = join(m, h), a_hl = join(h, l), a_hm = join(h, m);
#pragma unroll
        for (int ft = 0; ft < FT; ++ft) dacc[t][ft] = mfma_bf16(a_hl, b_lh[ft], dacc[t][ft]);
#pragma unroll
        for (int ft = 0; ft < FT; ++ft) dacc[t][ft] = mfma_bf16(a_mh, b_hm[ft], dacc[t][ft]);
#pragma unroll
        for (int ft = 0; ft < FT; ++ft) dacc[t][ft] = mfma_bf16(a_hm, b_hm[ft], dacc[t][ft]);
        __builtin_amdgcn_sched_barrier(0);
      }
    } else {  // probe only: keep the pointwise stage's results alive
#pragma unroll
      for (int t = 0; t < NT; ++t) asm volatile("" ::"v"(acc[t]));
#pragma unroll
      for (int j = 0; j < 4; ++j) asm volatile("" ::"v"(gx[j][0]), "v"(gx[j][1]));
    }
  }

  template <int LIK, bool LAST>
  __device__ __forceinline__ void run_tiles(const StepCtx& cx, const ModelConsts& mc, const float* s_w,
                                            const __bf16* planes) {
    const int lane = opaque_tid() & 63, n = lane & 15, q = lane >> 4;
    const int tb = cx.tile_begin, te = cx.tile_end;
    int fast_end = tb;
    if (cx.x_vec_ok && cx.y_vec_ok) fast_end = min(te, cx.n / 16);
    if (fast_end > tb) {
      // (the hardware issues the older of a SIMD's two waves first: without pacing it finishes its tiles well before the
      // younger and leaves it to run alone for a third of the loop)
      RowsA ra;
      load_a<true>(ra, cx, 16 * tb, n, q);
      for (int i = tb; i < fast_end; ++i) {
        RowsB rb;
        if (i > tb) keep_pace(cx, i - tb);
        compute_tile<LIK, LAST, true>(
            ra, rb, s_w, planes, cx, mc, 16 * i, n, q,
            [&] {  // this tile's rows for GEMM2, a pointwise stage away from their use
              load_b<true>(rb, cx, 16 * i, n, q);
              __builtin_amdgcn_sched_barrier(0);
            },
            [&] {  // the next tile's rows for GEMM1, half a contraction away
              load_a<true>(ra, cx, 16 * min(i + 1, fast_end - 1), n, q);
              __builtin_amdgcn_sched_barrier(0);
            });
      }
      __builtin_amdgcn_s_setprio(0);
    }
    for (int tile = max(tb, fast_end); tile < te; ++tile) tile_alone<LIK, LAST, false>(cx, mc, s_w, planes, tile, n, q);
    if (again_in_fp32(__builtin_isnan(db2acc), s_w, P)) {  // (the sum of all rows' loss gradients)
      zero_acc();
      for (int tile = tb; tile < te; ++tile) tile_alone<LIK, LAST, true>(cx, mc, s_w, planes, tile, n, q);
    }
  }
  template <int LIK, bool LAST, bool FP32>
  __device__ __forceinline__ void tile_alone(const StepCtx& cx, const ModelConsts& mc, const float* s_w,
                                             const __bf16* planes, int tile, int n, int q) {
    RowsA ra;
    RowsB rb;
    load_a<false>(ra, cx, tile * 16, n, q);
    load_b<false>(rb, cx, tile * 16, n, q);
    compute_tile<LIK, LAST, false, 3, FP32>(ra, rb, s_w, planes, cx, mc, tile * 16, n, q, [] {}, [] {});
  }

  // The workgroup record in LDS, in columns of four: the dW1 sums in accumulator order (a column is a lane's four
  // sums, which belong to four neighbouring parameters), everything else under its parameter number; unscaled
  // (record_values applies what compute_tile left out of delta).
  // the first of a column's four parameters
  static __device__ __forceinline__ int column_param(int col) {
    if (col >= D0 * D1 / 4) return 4 * col;
    const int lane = col & 63, tile = col >> 6, ft = tile % FT, t = tile / FT;
    const int f = 32 * (ft >> 1) + 2 * (lane & 15) + (ft & 1);
    return f * D1 + 16 * t + 4 * (lane >> 4);
  }
  // the values of a column, scaled: the factor 4 w2[c] of delta for dW1 and db1
  static __device__ __forceinline__ f4 record_values(f4 v, const float* s_w, int col) {
    static_assert(oB1 % D1 == 0 && D1 % 4 == 0 && oW2 % 4 == 0, "columns of dW1 and db1 lie within a row of W1");
    if (col >= oW2 / 4) return v;
    const f4 w2 = *reinterpret_cast<const f4*>(s_w + oW2 + column_param(col) % D1);
#pragma unroll
    for (int e = 0; e < 4; ++e) v[e] *= 4.0f * w2[e];
    return v;
  }
  // Add this wave's sums of hidden tile t to the record; `first` overwrites.  The waves of a workgroup do this
  // side by side, each on another tile, and move on to the next tile together: every element is added up in a
  // fixed order of waves.  (One wave after the other, in parameter order with its 16-way bank conflicts, took
  // most of the time of a step on few rows.)
  __device__ __forceinline__ void add_tile_partials(float* red, int tile, bool first) {
    const int lane = opaque_tid() & 63, n = lane & 15, q = lane >> 4;
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      if (t != tile) continue;  // wave-uniform
      // (16-byte columns, all reads in flight before the first addition: one sum after the other, 17 LDS round trips a
      // tile, took 9 us of a step)
      f4* dst = reinterpret_cast<f4*>(red) + t * FT * 64 + lane;
      f4 sum[FT];
#pragma unroll
      for (int ft = 0; ft < FT; ++ft) sum[ft] = dst[64 * ft];
#pragma unroll
      for (int ft = 0; ft < FT; ++ft) {
#pragma unroll
        for (int j = 0; j < 4; ++j) sum[ft][j] = first ? dacc[t][ft][j] : sum[ft][j] + dacc[t][ft][j];
      }
#pragma unroll
      for (int ft = 0; ft < FT; ++ft) dst[64 * ft] = sum[ft];
      // sums over the four row groups q in a fixed order, dw2 put together from the sums of g s and of g (see
      // prepare_step); lanes q < 2 end up with the sum of the one, lanes q >= 2 with that of the other
      float v = lane_fold32(db1acc[t], 2.0f * dw2acc[t] - db2acc);
      v = lane_fold16(v, v);
      if ((q & 1) == 0) {
        float* small = red + (q == 0 ? oB1 : oW2) + 16 * t + n;
        *small = first ? v : *small + v;
      }
    }
    if (tile == 0) {
      float b = db2acc;  // every lane n of a row group holds the same value
      b += __shfl_xor(b, 16);
      b += __shfl_xor(b, 32);
      double d = dl;  // held by the first lane of each bank
      d += shfl_xor_d(d, 4);
      d += shfl_xor_d(d, 8);
      d += shfl_xor_d(d, 16);
      d += shfl_xor_d(d, 32);
      if (lane == 0) {
        red[oB2] = first ? b : red[oB2] + b;
        double* dd = reinterpret_cast<double*>(red + P_AL);
        *dd = first ? d : *dd + d;
      }
    }
  }
};

}  // namespace bnn
