// Newton-Schulz iterations of a T x T tile (T = 128 or 256) with X in registers:
// T / 32 waves, wave w holding columns 32 w .. + 31 of X as T / 16 MFMA operands
// (T / 4 registers): lane l has column 32 w + l % 32, rows 16 ks + 8 (l / 32) .. + 7
// of operand ks. That is what Apply multiplies by, so Apply reads only B from
// LDS. The product's result layout (rows 8 q + 4 (l / 32) .. + 3 of a 32-row
// tile) turns into the operand layout by swapping register halves between
// lanes l and l + 32 (v_permlane32_swap), so X' replaces X without LDS. For
// X X^T every wave writes its columns to LDS, column by column (rows of T values
// of one X column), and all read row fragments with transposing reads. A and
// B replace X there: while X X^T accumulates no other matrix is live, and
// afterwards X is only needed in registers. A and B are symmetric and stored as
// their lower 32 x 32 tiles (lds_tiles.h).
//
// Each element sums its k terms in one accumulator in ascending order with the
// streamed kernels' MFMA, so the result has their bits (and torch's).
#pragma once

#include "lds_tiles.h"

namespace ns_reg {

// Wave W's share of a Gram product: row tiles ROW[0 .. NR - 1] as fragments, tile
// k (k < NTL) being (row tile ROW[I[k]], column tile ROW[J[k]]), row >= column.
template <int R0, int R1, int R2, int R3, int EXTRA>
struct CrossPart {  // rows R2, R3 by columns R0, R1, and (ROW[EXTRA], ROW[EXTRA])
  static constexpr int NR = 4, NTL = EXTRA < 0 ? 4 : 5;
  static constexpr int ROW[4] = {R0, R1, R2, R3};
  static constexpr int I[5] = {2, 2, 3, 3, EXTRA < 0 ? 0 : EXTRA}, J[5] = {0, 1, 0, 1, EXTRA < 0 ? 0 : EXTRA};
};
template <int R0, int R1, int R2, int R3>
struct DiagPart {  // (R1, R0) (R1, R1) (R3, R2) (R3, R3)
  static constexpr int NR = 4, NTL = 4;
  static constexpr int ROW[4] = {R0, R1, R2, R3};
  static constexpr int I[5] = {1, 1, 3, 3, 0}, J[5] = {0, 1, 2, 3, 0};
};

// 128 x 128: the 10 lower tiles over four waves, 3, 3, 2, 2.
struct Part128_0 {  // (0,0) (1,0) (1,1)
  static constexpr int NR = 2, NTL = 3, ROW[4] = {0, 1, 0, 0}, I[5] = {0, 1, 1, 0, 0}, J[5] = {0, 0, 1, 0, 0};
};
struct Part128_1 {  // (2,0) (2,1) (2,2)
  static constexpr int NR = 3, NTL = 3, ROW[4] = {0, 1, 2, 0}, I[5] = {2, 2, 2, 0, 0}, J[5] = {0, 1, 2, 0, 0};
};
struct Part128_2 {  // (3,0) (3,1)
  static constexpr int NR = 3, NTL = 2, ROW[4] = {0, 1, 3, 0}, I[5] = {2, 2, 0, 0, 0}, J[5] = {0, 1, 0, 0, 0};
};
struct Part128_3 {  // (3,2) (3,3)
  static constexpr int NR = 2, NTL = 2, ROW[4] = {2, 3, 0, 0}, I[5] = {1, 1, 0, 0, 0}, J[5] = {0, 1, 0, 0, 0};
};

template <int T, class F>
HM_DEV void with_part(int wave, F&& f) {
  if constexpr (T == 128) {
    switch (wave) {
      case 0: f(Part128_0{}); break;
      case 1: f(Part128_1{}); break;
      case 2: f(Part128_2{}); break;
      default: f(Part128_3{}); break;
    }
  } else {
    switch (wave) {
      case 0: f(CrossPart<0, 1, 2, 3, 0>{}); break;
      case 1: f(CrossPart<0, 1, 4, 5, 2>{}); break;
      case 2: f(CrossPart<4, 5, 6, 7, 2>{}); break;
      case 3: f(CrossPart<2, 3, 6, 7, 0>{}); break;
      case 4: f(CrossPart<2, 3, 4, 5, -1>{}); break;
      case 5: f(CrossPart<0, 1, 6, 7, -1>{}); break;
      case 6: f(DiagPart<0, 1, 2, 3>{}); break;
      default: f(DiagPart<4, 5, 6, 7>{}); break;
    }
  }
}

// Transposing read of a row-major T x T matrix in LDS (lds_pos layout): lane
// receives column c0 + l % 32 (c0 a multiple of 32), rows 16 ks + 8 (l / 32)
// .. + 7.
template <int T>
HM_DEV u32x4_t col_frag(const lds_u8* S, int c0, int ks, int tr_krow, int tr_col) {
  const int kr = 16 * ks + tr_krow, c = c0 + tr_col;
  const u32x2_t l2 = read_tr(S, lds_pos(kr, c >> 3, T / 8) + (c & 7) * 2);
  const u32x2_t u2 = read_tr(S, lds_pos(kr + 4, c >> 3, T / 8) + (c & 7) * 2);
  return u32x4_t{l2[0], l2[1], u2[0], u2[1]};
}

// Gram k-step K of part P, from X by columns (TRI false) or from the lower
// tiles of A.
template <int T, class P, bool TRI, int K, int R>
HM_DEV u32x4_t gram_frag(const lds_u8* S, int l32, int hi, int tr_krow, int tr_col) {
  if constexpr (TRI) return tri_frag<P::ROW[R], K>(S, l32, hi, tr_krow, tr_col);
  else return col_frag<T>(S, 32 * P::ROW[R], K, tr_krow, tr_col);
}
template <int T, class P, bool TRI, int K>
HM_DEV void gram_step(const lds_u8* S, int l32, int hi, int tr_krow, int tr_col, f32x16_t (&acc)[5]) {
  u32x4_t f[4];
  f[0] = gram_frag<T, P, TRI, K, 0>(S, l32, hi, tr_krow, tr_col);
  f[1] = gram_frag<T, P, TRI, K, 1>(S, l32, hi, tr_krow, tr_col);
  if constexpr (P::NR > 2) f[2] = gram_frag<T, P, TRI, K, 2>(S, l32, hi, tr_krow, tr_col);
  if constexpr (P::NR > 3) f[3] = gram_frag<T, P, TRI, K, 3>(S, l32, hi, tr_krow, tr_col);
#pragma unroll
  for (int k = 0; k < P::NTL; ++k) acc[k] = mfma(f[P::J[k]], f[P::I[k]], acc[k]);
}

template <int T, class P, bool TRI, int... K>
HM_DEV void gram_mma(const lds_u8* S, int lane, f32x16_t (&acc)[5], std::integer_sequence<int, K...>) {
  const int ln = opaque_lane(lane), l32 = ln & 31, hi = ln >> 5;
  const int tr_krow = tr_krow_of(ln), tr_col = tr_col_of(ln);
#pragma unroll
  for (int k = 0; k < P::NTL; ++k)
#pragma unroll
    for (int e = 0; e < 16; ++e) acc[k][e] = 0.f;
  (gram_step<T, P, TRI, K>(S, l32, hi, tr_krow, tr_col, acc), ...);
}

// Lane holds element 4 q + e of acc[k] at C[32 ROW[I[k]] + l32][32 ROW[J[k]] +
// 8 q + 4 hi + e].
template <class P>
HM_DEV void gram_store(lds_u8* C, int lane, const u32x2_t (&o)[5][4]) {
  const int ln = opaque_lane(lane), l32 = ln & 31, hi = ln >> 5;
#pragma unroll
  for (int k = 0; k < P::NTL; ++k)
#pragma unroll
    for (int q = 0; q < 4; ++q)
      *reinterpret_cast<lds_u32x2*>(C + tri_pos(P::ROW[P::I[k]], P::ROW[P::J[k]], l32, q) + hi * 8) = o[k][q];
}

template <int T, class P>
HM_DEV void gram_a(const lds_u8* X, int lane, u32x2_t (&o)[5][4]) {
  f32x16_t acc[5];
  gram_mma<T, P, false>(X, lane, acc, std::make_integer_sequence<int, T / 16>{});
#pragma unroll
  for (int k = 0; k < P::NTL; ++k)
#pragma unroll
    for (int q = 0; q < 4; ++q)
      o[k][q] = u32x2_t{pk_bf16(acc[k][4 * q], acc[k][4 * q + 1]), pk_bf16(acc[k][4 * q + 2], acc[k][4 * q + 3])};
}

template <int T, class P>
HM_DEV void gram_b(const lds_u8* A, int lane, float cb, float cc, u32x2_t (&o)[5][4]) {
  f32x16_t acc[5];
  gram_mma<T, P, true>(A, lane, acc, std::make_integer_sequence<int, T / 16>{});
  const int ln = opaque_lane(lane), l32 = ln & 31, hi = ln >> 5;
#pragma unroll
  for (int k = 0; k < P::NTL; ++k)
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const u32x2_t rv =
          *reinterpret_cast<lds_cu32x2*>(A + tri_pos(P::ROW[P::I[k]], P::ROW[P::J[k]], l32, q) + hi * 8);
      float y[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) y[e] = fmaf(cb, bf16_to_f32(half16(rv[e >> 1], e & 1)), cc * acc[k][4 * q + e]);
      o[k][q] = u32x2_t{pk_bf16(y[0], y[1]), pk_bf16(y[2], y[3])};
    }
}

// Operand layout <-> result layout of 16 rows of X: operand (c0, c1, c2, c3)
// of lane l holds rows 8 hi .. + 3 (c0, c1) and 8 hi + 4 .. + 7 (c2, c3);
// the result layout has rows 4 hi .. + 3 in (c0, c1) and 8 + 4 hi .. + 3 in
// (c2, c3). v_permlane32_swap exchanges the upper half wave of its first
// operand with the lower half of the second; it is its own inverse.
HM_DEV u32x4_t swap_halves(u32x4_t v) {
  const auto a = __builtin_amdgcn_permlane32_swap(v[0], v[2], false, false);
  const auto b = __builtin_amdgcn_permlane32_swap(v[1], v[3], false, false);
  return u32x4_t{a[0], b[0], a[1], b[1]};
}

// Apply: k-step K of row tiles R0 .. R0 + 3 of B against the wave's columns.
template <int R0, int K, int KS>
HM_DEV void apply_step(const lds_u8* B, int l32, int hi, int tr_krow, int tr_col, const u32x4_t (&x)[KS],
                       f32x16_t (&acc)[4]) {
  const u32x4_t f[4] = {tri_frag<R0, K>(B, l32, hi, tr_krow, tr_col), tri_frag<R0 + 1, K>(B, l32, hi, tr_krow, tr_col),
                        tri_frag<R0 + 2, K>(B, l32, hi, tr_krow, tr_col),
                        tri_frag<R0 + 3, K>(B, l32, hi, tr_krow, tr_col)};
#pragma unroll
  for (int t = 0; t < 4; ++t) acc[t] = mfma(f[t], x[K], acc[t]);
}

// Rows 32 R0 .. 32 R0 + 127 of X' for the wave's columns, in operand layout.
template <int R0, int KS, int... K>
HM_DEV void apply_rows(const lds_u8* B, int lane, float ca, int round_once, const u32x4_t (&x)[KS],
                       u32x4_t (&o)[8], std::integer_sequence<int, K...>) {
  const int ln = opaque_lane(lane), l32 = ln & 31, hi = ln >> 5;
  const int tr_krow = tr_krow_of(ln), tr_col = tr_col_of(ln);
  f32x16_t acc[4];
#pragma unroll
  for (int t = 0; t < 4; ++t)
#pragma unroll
    for (int e = 0; e < 16; ++e) acc[t][e] = 0.f;
  (apply_step<R0, K>(B, l32, hi, tr_krow, tr_col, x, acc), ...);
#pragma unroll
  for (int t = 0; t < 4; ++t)
#pragma unroll
    for (int s = 0; s < 2; ++s) {  // rows 16 s .. 16 s + 15 of the row tile
      const u32x4_t xv = swap_halves(x[2 * (R0 + t) + s]);
      u32x4_t r;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const float v0 = acc[t][8 * s + 2 * e], v1 = acc[t][8 * s + 2 * e + 1];
        const uint32_t bx = pk_bf16(v0, v1);
        const float b0 = round_once ? v0 : __uint_as_float(bx << 16);
        const float b1 = round_once ? v1 : __uint_as_float(bx & 0xffff0000u);
        r[e] = pk_bf16(fmaf(ca, __uint_as_float(xv[e] << 16), b0), fmaf(ca, __uint_as_float(xv[e] & 0xffff0000u), b1));
      }
      o[2 * t + s] = swap_halves(r);
    }
}

// `steps` >= 0 iterations on the row-major T x T tile in LDS (lds_pos layout, raw
// bf16 values; X0 = bf16(value inv)) by T / 32 waves; the result replaces it. L
// holds T * T * 2 bytes. Every thread calls it, after a barrier that publishes
// the tile; it ends with one that publishes the result.
template <int T>
HM_DEV void reg_iterations(lds_u8* L, float inv, int steps, float ca, float cb, float cc, int round_once) {
  static_assert(T == 128 || T == 256, "tile edge");
  constexpr int KS = T / 16, CH = T / 8;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);  // wave-uniform: scalar branches
  u32x4_t x[KS];
  {
    const int ln = opaque_lane(lane);
    const int tr_krow = tr_krow_of(ln), tr_col = tr_col_of(ln);
#pragma unroll
    for (int k = 0; k < KS; ++k) x[k] = scale8_rne(col_frag<T>(L, 32 * wave, k, tr_krow, tr_col), inv);
  }
  __syncthreads();  // every wave has its columns
#pragma unroll 1
  for (int it = 0; it < steps; ++it) {
    // ---- X by columns into LDS: row j of T holds column j of X --------------------
    {
      const int ln = opaque_lane(lane), l32 = ln & 31, hi = ln >> 5;
#pragma unroll
      for (int k = 0; k < KS; ++k)
        *reinterpret_cast<lds_u32x4*>(L + lds_pos(32 * wave + l32, 2 * k + hi, CH)) = x[k];
    }
    __syncthreads();
    // ---- A = bf16(X X^T), then B = bf16(c (A A^T) + b A), in its place -------------
    // (one dispatch on the wave-uniform index for both products and their
    // barriers, so a wave's tiles stay in registers; every wave passes the same
    // number of barriers)
    with_part<T>(wave, [&](auto part) {
      using P = decltype(part);
      u32x2_t o[5][4];
      gram_a<T, P>(L, lane, o);
      __syncthreads();  // every read of X is done
      gram_store<P>(L, lane, o);
      __syncthreads();
      gram_b<T, P>(L, lane, cb, cc, o);
      __syncthreads();  // every read of A is done
      gram_store<P>(L, lane, o);
    });
    __syncthreads();
    // ---- X' = bf16(bf16(B X) + a X) ------------------------------------------------
    u32x4_t o[KS / 8][8];
    apply_rows<0>(L, lane, ca, round_once, x, o[0], std::make_integer_sequence<int, KS>{});
    if constexpr (T == 256)
      apply_rows<4>(L, lane, ca, round_once, x, o[1], std::make_integer_sequence<int, KS>{});
#pragma unroll
    for (int k = 0; k < KS; ++k) x[k] = o[k / 8][k % 8];
    __syncthreads();  // every read of B is done
  }
  // ---- back to row-major: 4 x 4 transposes across lane quads -------------------------
  {
    const int ln = opaque_lane(lane), l32 = ln & 31, hi = ln >> 5, kq = ln & 3;
    const int c = 32 * wave + (l32 & ~3);
#pragma unroll
    for (int k = 0; k < KS; ++k) {
      const u32x4_t v = swap_halves(x[k]);
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const u32x2_t w = quad_transpose(u32x2_t{v[2 * h], v[2 * h + 1]}, kq);
        const int r = 16 * k + 8 * h + 4 * hi + kq;
        *reinterpret_cast<lds_u32x2*>(L + lds_pos(r, c >> 3, CH) + (c & 7) * 2) = w;
      }
    }
  }
  __syncthreads();
}

}  // namespace ns_reg
