// The MFMA layer of the 22 -> 40 -> 1 trajectory kernel: both contractions of a 16-row tile on
// v_mfma_f32_16x16x32_bf16 with every FP32 operand split into three bf16 parts (bnn_split_bf16.h; why the six
// products hh, hm, mh, hl, lh, mm of the parts are enough: bnn_mfma_wide_layer.h), the pointwise stage between
// them on the 40 real hidden units only.  The FP32 matrix instructions share their pipe with the vector
// instructions, the bf16 ones have one of their own, so what bounds the tile is its vector instructions (about 180 and
// 20 transcendentals; 31 matrix instructions): on 200 windows they are active 79 % of the SIMD cycles, the matrix pipe
// 38 %, some instruction 97 %.  Measured per tile and SIMD with two waves: 1260 cycles, against 1513
// for the same tile on FP32 matrix instructions with hidden 32 .. 39 on 4x4 blocks and 1696 for MfmaLayer; 0.565
// against 0.648 and 0.71 us (the denser mix runs at a lower clock: the card is limited by power).
//
// Lane l = 16 q + n, n = 4 cb + r, h8 = n >> 3, c8 = n & 7.
//   GEMM1  A = x_aug: lane (n, q) holds row n, k = 6 q + i in slots i < 6, zero in slots 6, 7 (24 k = 22 features,
//              the constant one that carries b1, a pad; as loaded from memory, split in registers)
//          hidden 0 .. 31: B = k W1_aug[6 q + i][16 t + n], one instruction per product
//          hidden 32 .. 39: eight of the sixteen columns would be empty, so they take another product of the same
//              A part: columns n < 8 and n >= 8 hold parts h and m of W1 (A = h and A = m: hh + mh and hm + mm), then
//              l and zero (A = h), h and zero (A = l).  Adding lane n ^ 8 sums the products; lanes n < 8 keep the
//              totals of rows 4 q, 4 q + 1 and lanes n >= 8 those of rows 4 q + 2, 4 q + 3: two values per lane
//              (sa, sb), rows ra = 4 q + 2 h8, ra + 1.
//   GEMM2  16 rows to contract and 32 k slots: two products share an instruction.  A = (u g)^T straight from the
//          C registers, slots 0 .. 3 and 4 .. 7 hold two parts of rows 4 q .. 4 q + 3.
//          features 0 .. 15: B = x_aug[row 4 q + j][n], [h | l] x [l | h], [m | h] x [h | m], [m | h] x [m | h]
//          features 16 .. 23: eight of sixteen columns again: [m | h] x [h | h] in columns n < 8 and x [m | m] in
//              columns n >= 8, and [h | l] x [l | h] and x zero
//          hidden 32 .. 39: lanes n < 8 fill the slots of rows 4 q, 4 q + 1, lanes n >= 8 those of 4 q + 2, 4 q + 3, the
//              others are zero; same B.  Rows m and m + 8 of the result are partial sums of hidden 32 + m.
//   B of GEMM2 is the transpose of what a lane has loaded: the wave writes the parts of its tile to LDS (16 rows x 24
//   bf16 each) and reads them back through ds_read_b64_tr_b16 (a row of 16 lanes reads 4 rows x 16 columns, every
//   lane receives the four rows of its column).
#pragma once

#include <hip/hip_runtime.h>

#include "bnn_device.h"
#include "bnn_kernel_common.h"
#include "bnn_mfma_layer.h"
#include "bnn_split_bf16.h"

namespace bnn {

template <int D0, int D1>
struct MfmaSplitLayer {
  static_assert(D0 == 22 && D1 == 40, "laid out for 22 features (24 with the bias and one pad) and 32 + 8 hidden units");
  static constexpr int KS = 6, KP = 3;  // k-steps of the wide GEMM1: 24 = 4 x 6
  static constexpr int NT = 2;          // 16-wide hidden tiles
  static constexpr int oB1 = D0 * D1, oW2 = oB1 + D1, oB2 = oW2 + D1, P = oB2 + 1;
  static constexpr int P_AL = (P + 3) / 4 * 4;
  // a wave's copy of the current tile in LDS: three parts of 16 rows x 24 bf16, then 16 bytes of zeros
  static constexpr int PART = 16 * 24;
  static constexpr int TILE_LDS = 3 * PART / 2 + 4;  // floats
  static constexpr float kExp2Scale = -2.88539008177792681472f;  // -2 / ln 2, kernel_helpers.h:37

  // per step (see MfmaLayer for the meaning of the scalings)
  bf8 w1[NT][3];       // hidden 0 .. 31: parts of k W1_aug[6 q + i][16 t + n]
  bf8 w5hm, w5l, w5h;  // hidden 32 .. 39: parts of k W1_aug[6 q + i][32 + c8]: h (n < 8) or m, l or zero, h or zero
  float w2g[NT], w2g5; // -2 w2[c] k2
  float k2v, y_0, rho, ratio;
  unsigned pad_h, pad_m, pad_l;  // zeros, see operand()
  // sums over rows
  f4 dacc_e[NT + 1];   // t < 2: hidden 16 t + 4 q + i, feature n; t = 2: rows m = 4 q + i, hidden 32 + (m & 7)
  f4 dacc_f[NT + 1];   // the same, feature 16 + c8, partial over the products of the column half h8
  float dw2s[NT];      // sum over the rows of group q of g' s, hidden 16 t + n
  float dw2s5;         // sum over the rows ra, ra + 1 of g' (s - 1/2), hidden 32 + c8
  float hs;            // sum over the rows of group q of g' / 2, added in the very order of dw2s: dw2 =
                       // 2 (dw2s - hs) is exactly zero where every s is 1/2 (all weights zero)
  double dl;

  struct TileIn {
    f2 xa[KP];   // GEMM1 operand: row n, k = 6 q + 2 i, + 1
    float y1;    // target of row 4 q + (n >> 2)
  };

  // The parts of k W1_aug, k = -2 / ln 2 (GEMM1 then yields the exp2 argument directly), in LDS as the lanes want
  // them: part, then [hidden tile][lane][8 slots].  The thread that updates a parameter splits it; what no parameter
  // occupies (pad feature, slots 6 and 7, columns 8 .. 15 of the third tile) is zero (clear_weights, once per launch).
  // (Split by every wave for itself from the FP32 weights, a step took 0.6 us longer.)
  static constexpr int W_PART = (NT + 1) * 64 * 8;
  static constexpr int W_PARTS = 3 * W_PART;
  static __device__ __forceinline__ void clear_weights(__bf16* parts, int tid, int threads) {
    for (int i = tid; i < W_PARTS / 8; i += threads) reinterpret_cast<f4*>(parts)[i] = f4{0.f, 0.f, 0.f, 0.f};
  }
  // where parameter p < oW2 goes: weight (k, c) of the first layer, or b1[c] as row k = D0
  static __device__ __forceinline__ int weight_offset(int p) {
    const int k = p / D1, c = p - k * D1;
    return ((c >> 4) * 64 + (k / KS) * 16 + (c & 15)) * 8 + k % KS;
  }
  static __device__ __forceinline__ void store_weight(__bf16* parts, int offset, float w) {
    __bf16* dst = parts + offset;
    split_scaled(w, kExp2Scale, dst[0], dst[W_PART], dst[2 * W_PART]);
  }

  template <int LIK>
  __device__ __forceinline__ void load_weights(const float* s_w, const __bf16* parts, const ModelConsts& mc) {
    const int lane = opaque_tid() & 63, n = lane & 15, q = lane >> 4, h8 = n >> 3, c8 = n & 7;
    const float k = LIK == 1 ? mc.scale_recp * mc.scale_recp : mc.scale_recp;
    const uint32_t k2_bits = (__builtin_bit_cast(uint32_t, k) + 0x00400000u) & 0x7F800000u;
    const float k2 = __builtin_bit_cast(float, k2_bits);
    ratio = __builtin_bit_cast(float, __builtin_amdgcn_readfirstlane(__builtin_bit_cast(
        int, k * __builtin_bit_cast(float, 0x7F000000u - k2_bits))));
    double w2lane = 0.0;
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      const int c = 16 * t + n;
#pragma unroll
      for (int part = 0; part < 3; ++part)
        w1[t][part] = *reinterpret_cast<const bf8*>(parts + part * W_PART + (64 * t + lane) * 8);
      const float w2c = s_w[oW2 + c];
      w2lane += (double)w2c;
      w2g[t] = -2.0f * w2c * k2;
    }
    {
      const int c = 32 + c8;
      const __bf16* third = parts + 64 * NT * 8;
      w5hm = *reinterpret_cast<const bf8*>(third + (h8 == 0 ? 0 : W_PART) + (16 * q + c8) * 8);
      w5l = *reinterpret_cast<const bf8*>(third + 2 * W_PART + lane * 8);
      w5h = *reinterpret_cast<const bf8*>(third + lane * 8);
      const float w2c = s_w[oW2 + c];
      // a lane's share of the constant covers hidden 32 + n once (lanes n < 8)
      if (h8 == 0) w2lane += (double)w2c;
      w2g5 = -2.0f * w2c * k2;
    }
    const double share = (w2lane - (n == 0 ? (double)s_w[oB2] : 0.0)) * (double)k2;
    y_0 = (float)share;
    const double rest = row16_allreduce_d(share - (double)y_0);
    rho = __builtin_bit_cast(float, __builtin_amdgcn_readfirstlane(__builtin_bit_cast(int, (float)rest)));
    k2v = __builtin_bit_cast(float, __builtin_amdgcn_readfirstlane(__builtin_bit_cast(int, k2)));
  }

  __device__ __forceinline__ void zero_acc() {
#pragma unroll
    for (int t = 0; t <= NT; ++t) dacc_e[t] = dacc_f[t] = f4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int t = 0; t < NT; ++t) dw2s[t] = 0.0f;
    dw2s5 = 0.0f;
    hs = 0.0f;
    dl = 0.0;
    // (not constants to the compiler: it would write them again for every tile)
    pad_h = pad_m = pad_l = 0u;
    asm volatile("" : "+v"(pad_h), "+v"(pad_m), "+v"(pad_l));
  }

  // rows past the end read as the last row (their gradient is masked to zero); any alignment
  __device__ __forceinline__ void load_tile_safe(TileIn& ti, const StepCtx& cx, int row0, int n, int q) const {
    const int last = cx.n - 1;
    const float* ra = cx.X + (size_t)min(row0 + n, last) * D0;
#pragma unroll
    for (int i = 0; i < KP; ++i) {
      const int k0 = KS * q + 2 * i;
      const int kc = k0 < D0 ? k0 : D0 - 2;
      f2 v = f2{ra[kc], ra[kc + 1]};
      if (k0 >= D0) v = f2{k0 == D0 ? 1.0f : 0.0f, 0.0f};
      ti.xa[i] = v;
    }
    ti.y1 = cx.y[min(row0 + 4 * q + (n >> 2), last)];
  }

  // four rows of a column of the tile's copy in LDS: lane (n, q) passes the address of the four columns
  // 4 (n & 3) .. of row 4 q + (n >> 2) and receives rows 4 q .. 4 q + 3 of column n
  static __device__ __forceinline__ bf4 read_transposed(const __bf16* p) {
    typedef short s4 __attribute__((ext_vector_type(4)));
    typedef __attribute__((address_space(3))) s4 lds_s4;
    return __builtin_bit_cast(bf4, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s4*)p));
  }

  // GEMM1 of a tile in FP32: x_aug, read again from memory (rows past the end: the last row), times W1_aug from the
  // FP32 weights in LDS, scaled afterwards (k times a large finite weight may be infinite).  The result as GEMM1 leaves
  // it, hidden 32 .. 39 in both column halves.
  __device__ __forceinline__ void gemm1_fp32(const StepCtx& cx, int row0, int n, int q, f4 (&acc)[NT], f4& acc5) const {
    const float* row = cx.X + (size_t)min(row0 + n, cx.n - 1) * D0;
    acc[0] = acc[1] = acc5 = f4{0.f, 0.f, 0.f, 0.f};
#pragma unroll 1
    for (int i = 0; i < KS; ++i) {
      const int k = KS * q + i;
      const float x = k < D0 ? row[min(k, D0 - 1)] : (k == D0 ? 1.0f : 0.0f);
      const float* w = cx.w_lds + min(k, D0) * D1;
      acc[0] = mfma_f32(x, k <= D0 ? w[n] : 0.0f, acc[0]);
      acc[1] = mfma_f32(x, k <= D0 ? w[16 + n] : 0.0f, acc[1]);
      acc5 = mfma_f32(x, k <= D0 ? w[32 + (n & 7)] : 0.0f, acc5);
    }
    acc[0] *= kExp2Scale;
    acc[1] *= kExp2Scale;
    acc5 *= kExp2Scale;
  }

  // One tile: the LDS copy, GEMM1, the pointwise stage, GEMM2.  `tile` is this wave's LDS buffer.
  // (GRAD == false: the forward half, for sums of the log-likelihood rows alone.  FP32: where a row sum is NaN,
  // GEMM1 in FP32.)
  template <int LIK, bool LAST, bool FULL, bool GRAD = true, bool FP32 = false>
  __device__ __forceinline__ void compute_tile(const TileIn& ti, float* tile, const StepCtx& cx,
                                               const ModelConsts& mc, int row0, int n, int q) {
    const int r = n & 3, h8 = n >> 3;
    // ---- the parts of the tile: GEMM1 operands and the wave's copy in LDS ----
    bf2 xh[KP], xm[KP], xl[KP];
#pragma unroll
    for (int i = 0; i < KP; ++i) split2(ti.xa[i], xh[i], xm[i], xl[i]);
    __bf16* parts = reinterpret_cast<__bf16*>(tile);
    if constexpr (GRAD) store_parts(parts, n, q, xh, xm, xl);
    const bf8 ah = operand(xh, pad_h), am = operand(xm, pad_m), al = operand(xl, pad_l);
    // ---- GEMM1, the small products first ----
    f4 acc[NT] = {f4{0.f, 0.f, 0.f, 0.f}, f4{0.f, 0.f, 0.f, 0.f}};
    f4 acc5 = f4{0.f, 0.f, 0.f, 0.f};
    acc5 = mfma_bf16(al, w5h, acc5);
    acc[0] = mfma_bf16(al, w1[0][0], acc[0]);
    acc[1] = mfma_bf16(al, w1[1][0], acc[1]);
    acc5 = mfma_bf16(ah, w5l, acc5);
    acc[0] = mfma_bf16(ah, w1[0][2], acc[0]);
    acc[1] = mfma_bf16(ah, w1[1][2], acc[1]);
    acc5 = mfma_bf16(am, w5hm, acc5);
    acc[0] = mfma_bf16(am, w1[0][1], acc[0]);
    acc[1] = mfma_bf16(am, w1[1][1], acc[1]);
    acc5 = mfma_bf16(ah, w5hm, acc5);
    acc[0] = mfma_bf16(am, w1[0][0], acc[0]);
    acc[1] = mfma_bf16(am, w1[1][0], acc[1]);
    acc[0] = mfma_bf16(ah, w1[0][1], acc[0]);
    acc[1] = mfma_bf16(ah, w1[1][1], acc[1]);
    acc[0] = mfma_bf16(ah, w1[0][0], acc[0]);
    acc[1] = mfma_bf16(ah, w1[1][0], acc[1]);
    // the GEMM2 operands from the LDS copy: issued here, used after the pointwise stage
    // (a part that several operands hold is read once for each: moving it would take vector instructions; the
    // second address is one the compiler does not know to be the first)
    bf8 be_lh, be_hm, be_mh, bf_hm, bf_lh;
    auto read_operands = [&] {
      const __bf16* rowp = parts + (4 * q + (n >> 2)) * 24;
      const __bf16* zeros = parts + 3 * PART;
      const __bf16* row2 = rowp + pad_h;
      const __bf16* row3 = rowp + pad_m;
      be_lh = join(read_transposed(rowp + 2 * PART + 4 * r), read_transposed(rowp + 4 * r));
      be_hm = join(read_transposed(row2 + 4 * r), read_transposed(row2 + PART + 4 * r));
      be_mh = join(read_transposed(row3 + PART + 4 * r), read_transposed(row3 + 4 * r));
      // features 16 .. 23: columns 0 .. 7 from lanes r = 0, 1 of a quad, columns 8 .. 15 from lanes r = 2, 3
      const __bf16* rowf = rowp + 16 + 4 * (r & 1);
      const __bf16* f_hm = rowf + (r < 2 ? 0 : PART);
      bf_hm = join(read_transposed(f_hm), read_transposed(f_hm + pad_l));
      bf_lh = join(read_transposed(r < 2 ? rowf + 2 * PART : zeros), read_transposed(r < 2 ? rowf : zeros));
    };
    if constexpr (GRAD) read_operands();
    __builtin_amdgcn_sched_barrier(0);
    // ---- hidden 32 .. 39: the products of the two column halves; lanes n < 8 keep rows 4 q, 4 q + 1 (registers
    //      0, 1), lanes n >= 8 rows 4 q + 2, 4 q + 3 (registers 2, 3) ----
    float sa, sb;
    {
      const float t0 = acc5[0] + dpp_move<0x128>(acc5[0]), t1 = acc5[1] + dpp_move<0x128>(acc5[1]);  // row_ror:8
      const float t2 = acc5[2] + dpp_move<0x128>(acc5[2]), t3 = acc5[3] + dpp_move<0x128>(acc5[3]);
      sa = h8 == 0 ? t0 : t2;
      sb = h8 == 0 ? t1 : t3;
    }
    // ---- pointwise stage (logistic form, see MfmaLayer::pointwise) ----
    float rz;
    auto row_sums = [&] {
      float yh[4] = {y_0, y_0, y_0, y_0};
#pragma unroll
      for (int t = 0; t < NT; ++t) {
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const float e = __builtin_amdgcn_exp2f(acc[t][j]);
          const float sg = __builtin_amdgcn_rcpf(1.0f + e);
          acc[t][j] = sg;
          yh[j] = __builtin_fmaf(w2g[t], sg, yh[j]);
        }
      }
      sa = __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(sa));
      sb = __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(sb));
      // hidden 32 .. 39 in the row sums: a lane holds two of its four rows
      asm("s_nop 1\n\t"
          "v_fmac_f32_dpp %[y0], %[a], %[w] quad_perm:[0,1,2,3] row_mask:0xf bank_mask:0x3\n\t"
          "v_fmac_f32_dpp %[y2], %[a], %[w] quad_perm:[0,1,2,3] row_mask:0xf bank_mask:0xc\n\t"
          "v_fmac_f32_dpp %[y1], %[b], %[w] quad_perm:[0,1,2,3] row_mask:0xf bank_mask:0x3\n\t"
          "v_fmac_f32_dpp %[y3], %[b], %[w] quad_perm:[0,1,2,3] row_mask:0xf bank_mask:0xc"
          : [y0] "+v"(yh[0]), [y1] "+v"(yh[1]), [y2] "+v"(yh[2]), [y3] "+v"(yh[3])
          : [a] "v"(sa), [b] "v"(sb), [w] "v"(w2g5));
      // (y - yhat - b2) k2 of the four rows 4 q + j, in bank j of one register
      rz = row16_reduce4(yh[0], yh[1], yh[2], yh[3]) + __builtin_fmaf(ti.y1, k2v, rho);
    };
    row_sums();
    if constexpr (FP32) {
      if (__builtin_amdgcn_ballot_w64(__builtin_isnan(rz)) != 0) {
        gemm1_fp32(cx, row0, n, q, acc, acc5);
        sa = h8 == 0 ? acc5[0] : acc5[2];
        sb = h8 == 0 ? acc5[1] : acc5[3];
        row_sums();
        if constexpr (GRAD) {
          // (a finite feature keeps finite parts in GEMM2; an infinite one makes NaN of its own weights' gradient)
#pragma unroll
          for (int i = 0; i < KP; ++i) split2_any(ti.xa[i], xh[i], xm[i], xl[i]);
          store_parts(parts, n, q, xh, xm, xl);
          read_operands();
        }
      }
    }
    float gz = rz, dz = rz;
    if (LIK == 0) {
      dz = rz * ratio;
      gz = dz * mc.g_scale * __builtin_amdgcn_rcpf(__builtin_fmaf(dz, dz, mc.df));
    }
    if (!FULL) gz = row0 + 4 * q + (n >> 2) < cx.n ? gz : 0.0f;  // mcmc_step_ffma.h:301 (the lane's bank holds that row)
    if (LAST) {
      // every lane holds the residual of its bank's row: the four rows of a lane group at once, stored and summed
      // by the first lane of each bank
      const int row = row0 + 4 * q + (n >> 2);
      const float lv = lik_value<LIK>(mc, LIK == 1 ? dz * (ratio * mc.scale) : dz);
      if (r == 0 && (FULL || row < cx.n)) {
        const float prev = cx.ell_prev ? cx.ell_prev[row] : 0.0f;
        if (cx.ell_new) cx.ell_new[row] = lv;
        dl += (double)(lv - prev);
      }
    }
    if constexpr (!GRAD) return;
    // dw2s += g s, hs += g / 2 (same order), dw2s5 += g (s - 1/2); then u g = (s - s^2) g in place.  g of row
    // 4 q + j is read from bank j of gz through a DPP row broadcast; for hidden 32 .. 39 lanes n < 8 take the
    // rows 4 q, 4 q + 1 (banks 0, 1) and lanes n >= 8 the rows 4 q + 2, 4 q + 3 (banks 2, 3).
    const float sa_c = sa - 0.5f, sb_c = sb - 0.5f;
    float uga = __builtin_fmaf(-sa, sa, sa), ugb = __builtin_fmaf(-sb, sb, sb);
    const float half = 0.5f;
#define BNN_BC(j) " row_newbcast:" #j " row_mask:0xf bank_mask:0xf\n\t"
    asm("s_nop 1\n\t"
        "v_fmac_f32_dpp %[d0], %[g], %[s00]" BNN_BC(0)
        "v_fmac_f32_dpp %[d1], %[g], %[s10]" BNN_BC(0)
        "v_fmac_f32_dpp %[hs], %[g], %[hf]" BNN_BC(0)
        "v_fmac_f32_dpp %[d0], %[g], %[s01]" BNN_BC(4)
        "v_fmac_f32_dpp %[d1], %[g], %[s11]" BNN_BC(4)
        "v_fmac_f32_dpp %[hs], %[g], %[hf]" BNN_BC(4)
        "v_fmac_f32_dpp %[d0], %[g], %[s02]" BNN_BC(8)
        "v_fmac_f32_dpp %[d1], %[g], %[s12]" BNN_BC(8)
        "v_fmac_f32_dpp %[hs], %[g], %[hf]" BNN_BC(8)
        "v_fmac_f32_dpp %[d0], %[g], %[s03]" BNN_BC(12)
        "v_fmac_f32_dpp %[d1], %[g], %[s13]" BNN_BC(12)
        "v_fmac_f32_dpp %[hs], %[g], %[hf]" BNN_BC(12)
        "v_fmac_f32_dpp %[d5], %[g], %[sa] row_newbcast:0 row_mask:0xf bank_mask:0x3\n\t"
        "v_fmac_f32_dpp %[d5], %[g], %[sa] row_newbcast:8 row_mask:0xf bank_mask:0xc\n\t"
        "v_fmac_f32_dpp %[d5], %[g], %[sb] row_newbcast:4 row_mask:0xf bank_mask:0x3\n\t"
        "v_fmac_f32_dpp %[d5], %[g], %[sb] row_newbcast:12 row_mask:0xf bank_mask:0xc"
        : [d0] "+v"(dw2s[0]), [d1] "+v"(dw2s[1]), [hs] "+v"(hs), [d5] "+v"(dw2s5)
        : [g] "v"(gz), [hf] "v"(half), [s00] "v"(acc[0][0]), [s01] "v"(acc[0][1]), [s02] "v"(acc[0][2]),
          [s03] "v"(acc[0][3]), [s10] "v"(acc[1][0]), [s11] "v"(acc[1][1]), [s12] "v"(acc[1][2]),
          [s13] "v"(acc[1][3]), [sa] "v"(sa_c), [sb] "v"(sb_c));
    float ug[NT][4];
#pragma unroll
    for (int t = 0; t < NT; ++t) {
#pragma unroll
      for (int j = 0; j < 4; ++j) ug[t][j] = __builtin_fmaf(-acc[t][j], acc[t][j], acc[t][j]);
    }
    asm("s_nop 1\n\t"
        "v_mul_f32_dpp %[u00], %[g], %[u00]" BNN_BC(0)
        "v_mul_f32_dpp %[u10], %[g], %[u10]" BNN_BC(0)
        "v_mul_f32_dpp %[u01], %[g], %[u01]" BNN_BC(4)
        "v_mul_f32_dpp %[u11], %[g], %[u11]" BNN_BC(4)
        "v_mul_f32_dpp %[u02], %[g], %[u02]" BNN_BC(8)
        "v_mul_f32_dpp %[u12], %[g], %[u12]" BNN_BC(8)
        "v_mul_f32_dpp %[u03], %[g], %[u03]" BNN_BC(12)
        "v_mul_f32_dpp %[u13], %[g], %[u13]" BNN_BC(12)
        "v_mul_f32_dpp %[ua], %[g], %[ua] row_newbcast:0 row_mask:0xf bank_mask:0x3\n\t"
        "v_mul_f32_dpp %[ua], %[g], %[ua] row_newbcast:8 row_mask:0xf bank_mask:0xc\n\t"
        "v_mul_f32_dpp %[ub], %[g], %[ub] row_newbcast:4 row_mask:0xf bank_mask:0x3\n\t"
        "v_mul_f32_dpp %[ub], %[g], %[ub] row_newbcast:12 row_mask:0xf bank_mask:0xc"
        : [u00] "+v"(ug[0][0]), [u01] "+v"(ug[0][1]), [u02] "+v"(ug[0][2]), [u03] "+v"(ug[0][3]),
          [u10] "+v"(ug[1][0]), [u11] "+v"(ug[1][1]), [u12] "+v"(ug[1][2]), [u13] "+v"(ug[1][3]),
          [ua] "+v"(uga), [ub] "+v"(ugb)
        : [g] "v"(gz));
#undef BNN_BC
    __builtin_amdgcn_sched_barrier(0);
    // ---- GEMM2 ----
    auto contract = [&](int t, bf4 h, bf4 m, bf4 l) {
      const bf8 hl = join(h, l), mh = join(m, h);
      dacc_e[t] = mfma_bf16(hl, be_lh, dacc_e[t]);
      dacc_f[t] = mfma_bf16(hl, bf_lh, dacc_f[t]);
      dacc_e[t] = mfma_bf16(mh, be_hm, dacc_e[t]);
      dacc_f[t] = mfma_bf16(mh, bf_hm, dacc_f[t]);
      dacc_e[t] = mfma_bf16(mh, be_mh, dacc_e[t]);
    };
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      bf4 h, m, l;
      split4(f4{ug[t][0], ug[t][1], ug[t][2], ug[t][3]}, h, m, l);
      contract(t, h, m, l);
    }
    {
      bf2 h, m, l;
      split2(f2{uga, ugb}, h, m, l);
      contract(NT, rows_of_half(h, h8), rows_of_half(m, h8), rows_of_half(l, h8));
    }
    __builtin_amdgcn_sched_barrier(0);
  }
  // slots 6 and 7 from a register that holds zeros (one per part, so that an operand's four registers stay together
  // from tile to tile and nothing is moved)
  static __device__ __forceinline__ bf8 operand(const bf2 (&p)[KP], unsigned zeros) {
    typedef unsigned u4 __attribute__((ext_vector_type(4)));
    return __builtin_bit_cast(bf8, u4{__builtin_bit_cast(unsigned, p[0]), __builtin_bit_cast(unsigned, p[1]),
                                      __builtin_bit_cast(unsigned, p[2]), zeros});
  }
  // lane (n, q)'s parts in the wave's copy of the tile
  static __device__ __forceinline__ void store_parts(__bf16* parts, int n, int q, const bf2 (&h)[KP], const bf2 (&m)[KP],
                                                     const bf2 (&l)[KP]) {
    bf2* dst = reinterpret_cast<bf2*>(parts + n * 24 + KS * q);
#pragma unroll
    for (int i = 0; i < KP; ++i) {
      dst[i] = h[i];
      dst[PART / 2 + i] = m[i];
      dst[2 * (PART / 2) + i] = l[i];
    }
  }
  // two values in the slots of rows 0, 1 (lanes n < 8) or 2, 3 of the four, zeros in the others
  static __device__ __forceinline__ bf4 rows_of_half(bf2 v, int h8) {
    const unsigned b = __builtin_bit_cast(unsigned, v);
    const unsigned lo = h8 == 0 ? b : 0u, hi = h8 == 0 ? 0u : b;
    return __builtin_bit_cast(bf4, ((unsigned long long)hi << 32) | lo);
  }

  // ---- explicitly prefetched loop (see MfmaLayer::prefetch_loop): loads issued from inline assembly two tiles
  //      ahead into three rotating register sets, explicit waits ----
  static constexpr int N_LOADS = 3;
  struct TileRaw {
    f4 xa01;   // GEMM1 operand, k-pairs 0 and 1
    TileIn t;  // t.xa[2]: k-pair 2 (the (1, 0) constant in lane group q = 3); t.xa[0 .. 1] from xa01 at use
  };
  template <int N>
  static __device__ __forceinline__ void wait_tile(TileRaw& r) {
    asm volatile("s_waitcnt vmcnt(%[cnt])"
                 : "+v"(r.xa01), "+v"(r.t.xa[KP - 1]), "+v"(r.t.y1)
                 : [cnt] "n"(N)
                 : "memory");
  }
  struct LoadPlan {
    unsigned oa, ol, oy;
    unsigned long long mask_a;
  };
  static __device__ __forceinline__ LoadPlan load_plan(int n, int q) {
    LoadPlan lp;
    lp.oa = (unsigned)((n * D0 + KS * q) * 4);
    lp.ol = lp.oa + 2 * (KP - 1) * 4;
    lp.oy = (unsigned)((4 * q + (n >> 2)) * 4);
    const bool a_const = KS * q + 2 * (KP - 1) >= D0;
    lp.mask_a = __builtin_amdgcn_ballot_w64(!a_const);
    return lp;
  }
  static __device__ __forceinline__ void preset(TileRaw& r) { r.t.xa[KP - 1] = f2{1.0f, 0.0f}; }
  // exactly N_LOADS loads of one full tile (see MfmaLayer::issue_tile for the s_nop, EXEC and early-clobber)
  static __device__ __forceinline__ void issue_tile(TileRaw& r, const StepCtx& cx, const LoadPlan& lp, int tile) {
    const float* bx = cx.X + (size_t)tile * (16 * D0);
    const float* by = cx.y + (size_t)tile * 16;
    unsigned long long exec_save;
    asm volatile(
        "s_mov_b64 %[sv], exec\n\t"
        "s_nop 3\n\t"
        "global_load_dwordx4 %[xa01], %[oa], %[bx]\n\t"
        "global_load_dword %[y1], %[oy], %[by]\n\t"
        "s_and_b64 exec, %[sv], %[ma]\n\t"
        "global_load_dwordx2 %[xa2], %[ol], %[bx]\n\t"
        "s_mov_b64 exec, %[sv]"
        : [xa01] "=&v"(r.xa01), [xa2] "+v"(r.t.xa[KP - 1]), [y1] "=&v"(r.t.y1), [sv] "=&s"(exec_save)
        : [oa] "v"(lp.oa), [ol] "v"(lp.ol), [oy] "v"(lp.oy), [bx] "s"(bx), [by] "s"(by), [ma] "s"(lp.mask_a)
        : "memory", "scc");
  }

  static __device__ __forceinline__ int fast_end_of(const StepCtx& cx) {
    int fast_end = cx.tile_begin;
    if (cx.x_vec_ok && cx.y_vec_ok) fast_end = min(cx.tile_end, cx.n / 16);
    return fast_end;
  }

  // A wave walks its run of tiles forwards in one gradient evaluation and backwards in the next (cx.back,
  // cx.back_next): what it read last -- what the caches most likely still hold when the rows of all chains in
  // flight exceed them -- is what it reads first.  The partial sums of a backward evaluation are added in the
  // opposite order, so the direction is a function of the leapfrog step alone, and the last step of a trajectory,
  // whose gradient a chain carries into its next transition (and a resumed chain computes afresh), always goes
  // forwards.
  TileRaw pa, pb;  // the first two tiles of the next evaluation (see MfmaLayer)
  // tile number k of an evaluation's walk over [tb, te)
  static __device__ __forceinline__ int walk(int tb, int te, int k, int back) { return back ? te - 1 - k : tb + k; }
  // A run of one or two tiles stays in the registers from one evaluation to the next, taken forwards every time: with
  // so few tiles a reload would have nothing to hide behind (about 1000 cycles of a step of 15000).
  static constexpr int KEPT = 2;
  __device__ __forceinline__ void prime(const StepCtx& cx) {
    const int tb = cx.tile_begin, te = fast_end_of(cx);
    if (te <= tb) return;
    const int lane = opaque_tid() & 63;
    const LoadPlan lp = load_plan(lane & 15, lane >> 4);
    const int back = te - tb <= KEPT ? 0 : __builtin_amdgcn_readfirstlane(cx.back);
    preset(pa);
    preset(pb);
    issue_tile(pa, cx, lp, __builtin_amdgcn_readfirstlane(walk(tb, te, 0, back)));
    issue_tile(pb, cx, lp, __builtin_amdgcn_readfirstlane(walk(tb, te, tb + 1 < te ? 1 : 0, back)));
    wait_tile<0>(pa);
    wait_tile<0>(pb);
  }

  template <int LIK, bool LAST, bool GRAD>
  __device__ __forceinline__ void prefetch_loop(const StepCtx& cx, const ModelConsts& mc, int tb, int te, int n,
                                                int q) {
    float* tile = cx.tile_lds;
    if (te - tb <= KEPT) {
      // (a run of one tile has it in both register sets)
#pragma unroll 1
      for (int i = tb; i < te; ++i) {
        pa.t.xa[0] = f2{pa.xa01[0], pa.xa01[1]};
        pa.t.xa[1] = f2{pa.xa01[2], pa.xa01[3]};
        compute_tile<LIK, LAST, true, GRAD>(pa.t, tile, cx, mc, i * 16, n, q);
        const TileRaw done = pa;
        pa = pb;
        pb = done;
      }
      return;
    }
    const LoadPlan lp = load_plan(n, q);
    // the loads run two tiles ahead of the arithmetic along the walk, into the next evaluation's (which goes
    // the other way) at the end of this one's
    const int back = __builtin_amdgcn_readfirstlane(cx.back);
    const int back_next = __builtin_amdgcn_readfirstlane(cx.back_next);
    const int len = te - tb;
    int nk = 2, nback = back;  // (len > KEPT)
    auto issue = [&](TileRaw& r) {
      issue_tile(r, cx, lp, __builtin_amdgcn_readfirstlane(walk(tb, te, nk, nback)));
      if (++nk == len) {
        nk = 0;
        nback = back_next;
      }
    };
    auto compute = [&](TileRaw& r, int i) {  // i: tb + position in the walk
      r.t.xa[0] = f2{r.xa01[0], r.xa01[1]};
      r.t.xa[1] = f2{r.xa01[2], r.xa01[3]};
      compute_tile<LIK, LAST, true, GRAD>(r.t, tile, cx, mc, walk(tb, te, i - tb, back) * 16, n, q);
    };
    TileRaw& A = pa;
    TileRaw& B = pb;
    TileRaw C;
    preset(C);
    int i = tb;
    for (; i + 3 <= te; i += 3) {
      issue(C);
      wait_tile<2 * N_LOADS>(A);
      compute(A, i);
      issue(A);
      wait_tile<2 * N_LOADS>(B);
      compute(B, i + 1);
      issue(B);
      wait_tile<2 * N_LOADS>(C);
      compute(C, i + 2);
      keep_pace(cx, i + 3 - tb);
    }
    if (cx.progress != nullptr) __builtin_amdgcn_s_setprio(0);
    const int left = te - i;
    if (left >= 1) {
      issue(C);
      wait_tile<2 * N_LOADS>(A);
      compute(A, i);
      if (left == 2) {
        issue(A);
        wait_tile<2 * N_LOADS>(B);
        compute(B, i + 1);
      }
    }
    wait_tile<0>(A);
    wait_tile<0>(B);
    wait_tile<0>(C);
    if (left == 1) {
      A = B;
      B = C;
    } else if (left == 2) {
      const TileRaw first = C;
      B = A;
      A = first;
    }
  }

  template <int LIK, bool LAST, bool GRAD = true>
  __device__ __forceinline__ void run_tiles(const StepCtx& cx, const ModelConsts& mc) {
    const int lane = opaque_tid() & 63, n = lane & 15, q = lane >> 4;
    const int tb = cx.tile_begin, te = cx.tile_end;
    const int fast_end = fast_end_of(cx);
    if (lane < 4) cx.tile_lds[3 * PART / 2 + lane] = 0.0f;
    if (fast_end > tb) prefetch_loop<LIK, LAST, GRAD>(cx, mc, tb, fast_end, n, q);
    // ragged tail tile, or unaligned caller buffers: one tile at a time
    for (int tile = max(tb, fast_end); tile < te; ++tile) tile_alone<LIK, LAST, GRAD, false>(cx, mc, tile, n, q);
    // (hs is the sum of all rows' loss gradients, dl of their log-likelihoods)
    if (again_in_fp32(GRAD ? __builtin_isnan(hs) : __builtin_isnan(dl), cx.w_lds, P)) {
      zero_acc();
      for (int tile = tb; tile < te; ++tile) tile_alone<LIK, LAST, GRAD, true>(cx, mc, tile, n, q);
    }
  }
  template <int LIK, bool LAST, bool GRAD, bool FP32>
  __device__ __forceinline__ void tile_alone(const StepCtx& cx, const ModelConsts& mc, int tile, int n, int q) {
    TileIn ti;
    load_tile_safe(ti, cx, tile * 16, n, q);
    compute_tile<LIK, LAST, false, GRAD, FP32>(ti, cx.tile_lds, cx, mc, tile * 16, n, q);
  }

  // after fold4(x0, y0, x1, y1) row q of lanes holds the sum over the four rows of lanes of x0 (q = 0),
  // x1 (q = 1), y0 (q = 2), y1 (q = 3), added as (q0 + q2) + (q1 + q3)
  static __device__ __forceinline__ float fold4(float x0, float y0, float x1, float y1) {
    return lane_fold16(lane_fold32(x0, y0), lane_fold32(x1, y1));
  }

  // ---- the wave's partial sums in LDS: the table of MfmaLayer (48-float rows: row f < D0 feature f, row D0
  //      the bias, row 24 the layer-2 weights, row 25 the log-likelihood difference; column = hidden unit,
  //      column D1 of the bias row holds the sum for b2) ----
  static constexpr int ROW = 48;
  static constexpr int W2_ROW = 24, DL_ROW = 25;
  static constexpr int LDS_SLOT = (DL_ROW + 1) * ROW;
  static constexpr int DL_INDEX = DL_ROW * ROW;
  static __device__ __forceinline__ int slot_index(int p) {
    if (p < oW2) return (p / D1) * ROW + p % D1;
    if (p < oB2) return W2_ROW * ROW + (p - oW2);
    return D0 * ROW + D1;
  }
  template <int LIK>
  __device__ __forceinline__ float finish(int p, float v, const float* s_w) const {
    const float gr = LIK == 1 ? ratio : 1.0f;
    if (p < oW2) return v * (4.0f * gr * s_w[oW2 + p % D1]);
    return v * gr;  // layer-2 weights and b2
  }

  template <int LIK>
  __device__ __forceinline__ void write_partials(float* slot, const float*, bool last) {
    const int lane = opaque_tid() & 63, n = lane & 15, q = lane >> 4, c8 = n & 7;
    // The lane swaps below read this accumulator from inside assembly statements, where the compiler does not count
    // the wait states a vector instruction needs after a matrix instruction wrote its operand (up to 11).  Once per
    // step: sixteen wait states here cover whatever the tile loop ended on; the accumulator is an operand, so that no
    // swap can be scheduled before them.
    asm volatile("s_nop 15" : "+v"(dacc_e[NT]));
    // ---- hidden 0 .. 31: lane (n, q), component i: c = 16 t + 4 q + i, f = n and f = 16 + c8 (lanes n and n ^ 8
    //      store the same bits to the same place) ----
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      *reinterpret_cast<f4*>(slot + n * ROW + 16 * t + 4 * q) = dacc_e[t];
      f4 v = dacc_f[t];
#pragma unroll
      for (int i = 0; i < 4; ++i) v[i] += dpp_move<0x128>(v[i]);  // row_ror:8
      *reinterpret_cast<f4*>(slot + (16 + c8) * ROW + 16 * t + 4 * q) = v;
    }
    // ---- hidden 32 .. 39: rows m and m + 8 of the result, two lane groups q apart ----
    {
      f4 vf = dacc_f[NT];
#pragma unroll
      for (int i = 0; i < 4; ++i) vf[i] += dpp_move<0x128>(vf[i]);
      const int c = 32 + 4 * (q & 1) + (q >> 1);
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        slot[n * ROW + c + 2 * h] = lane_fold32(dacc_e[NT][2 * h], dacc_e[NT][2 * h + 1]);
        slot[(16 + c8) * ROW + c + 2 * h] = lane_fold32(vf[2 * h], vf[2 * h + 1]);
      }
    }
    // ---- dw2 = sum g h = 2 sum g (s - 1/2): hidden 0 .. 31 as 2 (dw2s - hs), hidden 32 .. 39 as 2 dw2s5;
    //      db2 = sum g = 2 hs.  Row q of lanes ends with: q = 0 hidden n, q = 2 hidden 16 + n, q = 1 and 3
    //      hidden 32 + c8 (lanes n and n ^ 8, rows 1 and 3 store the same bits to the same place) ----
    {
      float d5s = dw2s5;
      d5s += dpp_move<0x128>(d5s);
      const float v = fold4(2.0f * (dw2s[0] - hs), 2.0f * (dw2s[1] - hs), 2.0f * d5s, 2.0f * d5s);
      const int col = q == 0 ? n : (q == 2 ? 16 + n : 32 + (n & 7));
      slot[W2_ROW * ROW + col] = v;
      const float g2 = fold4(hs, hs, hs, hs);  // every lane: the sum over the wave's rows of g / 2
      if (lane == 0) slot[D0 * ROW + D1] = 2.0f * g2;
    }
    if (last) {
      double d = dl;  // held by the first lane of each bank
      d += shfl_xor_d(d, 4);
      d += shfl_xor_d(d, 8);
      d += shfl_xor_d(d, 16);
      d += shfl_xor_d(d, 32);
      if (lane == 0) {
        const uint64_t bits = double_to_bits(d);
        slot[DL_INDEX] = __builtin_bit_cast(float, (uint32_t)bits);
        slot[DL_INDEX + 1] = __builtin_bit_cast(float, (uint32_t)(bits >> 32));
      }
    }
  }
};

}  // namespace bnn
