// Newton-Schulz for NS tiles with mp == np == 256, all iterations in one
// launch: a workgroup of eight waves (two per SIMD, one workgroup per CU) keeps
// X in registers and passes it and A / B through 128 KiB of LDS, so HBM sees
// one read and one write of the tile. Rounding points as in the three-kernel
// path (XXT.py:55-75, ba_plus_cAA.py:58-85, fused_bmm_add.py:65-88):
//
//   X0 = bf16(x inv)
//   A  = bf16(X X^T)              lower 32 x 32 tiles only
//   B  = bf16(c (A A^T) + b A)    lower 32 x 32 tiles only
//   X' = bf16(bf16(B X) + a X)
//
// What bounds it: the three streamed products move 7 matrices per tile and
// iteration (0.9 MB for 67 MFLOP of needed products, 75 FLOP/B) and are bound
// by that traffic and by 15 launches; here a tile needs 0.26 MB for all five
// iterations, and the MFMAs (2,176 v_mfma_f32_32x32x16_bf16 per iteration) and
// the LDS reads of their operands bound it.
//
// X (256 x 256): wave w holds columns 32 w .. + 31 as 16 MFMA operands (64
// registers): lane l has column 32 w + l % 32, rows 16 ks + 8 (l / 32) .. + 7
// of operand ks. That is what Apply multiplies by, so Apply reads only B from
// LDS. The product's result layout (rows 8 q + 4 (l / 32) .. + 3 of a 32-row
// tile) turns into the operand layout by swapping register halves between
// lanes l and l + 32 (v_permlane32_swap), so X' replaces X without LDS. For
// X X^T every wave writes its columns to LDS, column by column (512-byte rows
// of one X column), and all read row fragments with transposing reads. A and
// B replace X there: while X X^T accumulates no other matrix is live, and
// afterwards X is only needed in registers. A and B are stored as their 36
// lower 32 x 32 tiles (72 KiB), as in ns5_lds.hip.
//
// The Gram products' 36 tiles are split 5, 5, 5, 5, 4, 4, 4, 4 over the waves
// (9 per SIMD, wave w sharing SIMD w % 4 with wave w + 4), each wave working
// from four row fragments per k-step. Each element sums its k terms in one
// accumulator in ascending order with the streamed kernels' MFMA, so the
// result has their bits (and torch's).
#include "tile_step.h"

namespace {

constexpr int T = 256;          // tile edge
constexpr int NT = 512;         // threads: eight waves
constexpr int CH = T / 8;       // 16-byte chunks per row
constexpr int KS = T / 16;      // MFMA k-steps
constexpr int LDS_BYTES = T * T * 2;
// 8-element vectors whose loads are in flight per thread in the step's memory
// passes (grad and momentum: 16 VGPRs each, parameters: 8 or 4)
constexpr int GAT_BATCH = 4, UNT_BATCH = 8;

// Wave W's share of a Gram product: row tiles ROW[0 .. 3] as fragments, tile k
// (k < NTL) being (row tile ROW[I[k]], column tile ROW[J[k]]), row >= column.
template <int R0, int R1, int R2, int R3, int EXTRA>
struct CrossPart {  // rows R2, R3 by columns R0, R1, and (ROW[EXTRA], ROW[EXTRA])
  static constexpr int NTL = EXTRA < 0 ? 4 : 5;
  static constexpr int ROW[4] = {R0, R1, R2, R3};
  static constexpr int I[5] = {2, 2, 3, 3, EXTRA < 0 ? 0 : EXTRA}, J[5] = {0, 1, 0, 1, EXTRA < 0 ? 0 : EXTRA};
};
template <int R0, int R1, int R2, int R3>
struct DiagPart {  // (R1, R0) (R1, R1) (R3, R2) (R3, R3)
  static constexpr int NTL = 4;
  static constexpr int ROW[4] = {R0, R1, R2, R3};
  static constexpr int I[5] = {1, 1, 3, 3, 0}, J[5] = {0, 1, 2, 3, 0};
};

template <class F>
HM_DEV void with_part(int wave, F&& f) {
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

// Transposing read of a row-major T x T matrix in LDS (lds_pos layout): lane
// receives column c0 + l % 32 (c0 a multiple of 32), rows 16 ks + 8 (l / 32)
// .. + 7.
HM_DEV u32x4_t col_frag(const lds_u8* S, int c0, int ks, int tr_krow, int tr_col) {
  const int kr = 16 * ks + tr_krow, c = c0 + tr_col;
  const u32x2_t l2 = read_tr(S, lds_pos(kr, c >> 3, CH) + (c & 7) * 2);
  const u32x2_t u2 = read_tr(S, lds_pos(kr + 4, c >> 3, CH) + (c & 7) * 2);
  return u32x4_t{l2[0], l2[1], u2[0], u2[1]};
}

// Gram k-step K of part P, from X by columns (TRI false) or from the lower
// tiles of A.
template <class P, bool TRI, int K>
HM_DEV void gram_step(const lds_u8* S, int l32, int hi, int tr_krow, int tr_col, f32x16_t (&acc)[5]) {
  u32x4_t f[4];
  if constexpr (TRI) {
    f[0] = tri_frag<P::ROW[0], K>(S, l32, hi, tr_krow, tr_col);
    f[1] = tri_frag<P::ROW[1], K>(S, l32, hi, tr_krow, tr_col);
    f[2] = tri_frag<P::ROW[2], K>(S, l32, hi, tr_krow, tr_col);
    f[3] = tri_frag<P::ROW[3], K>(S, l32, hi, tr_krow, tr_col);
  } else {
#pragma unroll
    for (int r = 0; r < 4; ++r) f[r] = col_frag(S, 32 * P::ROW[r], K, tr_krow, tr_col);
  }
#pragma unroll
  for (int k = 0; k < P::NTL; ++k) acc[k] = mfma(f[P::J[k]], f[P::I[k]], acc[k]);
}

template <class P, bool TRI, int... K>
HM_DEV void gram_mma(const lds_u8* S, int lane, f32x16_t (&acc)[5], std::integer_sequence<int, K...>) {
  const int ln = opaque_lane(lane), l32 = ln & 31, hi = ln >> 5;
  const int tr_krow = tr_krow_of(ln), tr_col = tr_col_of(ln);
#pragma unroll
  for (int k = 0; k < P::NTL; ++k)
#pragma unroll
    for (int e = 0; e < 16; ++e) acc[k][e] = 0.f;
  (gram_step<P, TRI, K>(S, l32, hi, tr_krow, tr_col, acc), ...);
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

template <class P>
HM_DEV void gram_a(const lds_u8* X, int lane, u32x2_t (&o)[5][4]) {
  f32x16_t acc[5];
  gram_mma<P, false>(X, lane, acc, std::make_integer_sequence<int, KS>{});
#pragma unroll
  for (int k = 0; k < P::NTL; ++k)
#pragma unroll
    for (int q = 0; q < 4; ++q)
      o[k][q] = u32x2_t{pk_bf16(acc[k][4 * q], acc[k][4 * q + 1]), pk_bf16(acc[k][4 * q + 2], acc[k][4 * q + 3])};
}

template <class P>
HM_DEV void gram_b(const lds_u8* A, int lane, float cb, float cc, u32x2_t (&o)[5][4]) {
  f32x16_t acc[5];
  gram_mma<P, true>(A, lane, acc, std::make_integer_sequence<int, KS>{});
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
template <int R0, int K>
HM_DEV void apply_step(const lds_u8* B, int l32, int hi, int tr_krow, int tr_col, const u32x4_t (&x)[KS],
                       f32x16_t (&acc)[4]) {
  const u32x4_t f[4] = {tri_frag<R0, K>(B, l32, hi, tr_krow, tr_col), tri_frag<R0 + 1, K>(B, l32, hi, tr_krow, tr_col),
                        tri_frag<R0 + 2, K>(B, l32, hi, tr_krow, tr_col),
                        tri_frag<R0 + 3, K>(B, l32, hi, tr_krow, tr_col)};
#pragma unroll
  for (int t = 0; t < 4; ++t) acc[t] = mfma(f[t], x[K], acc[t]);
}

// Rows 32 R0 .. 32 R0 + 127 of X' for the wave's columns, in operand layout.
template <int R0, int... K>
HM_DEV void apply_half(const lds_u8* B, int lane, float ca, int round_once, const u32x4_t (&x)[KS],
                       u32x4_t (&o)[KS / 2], std::integer_sequence<int, K...>) {
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

// `steps` >= 0 iterations on the row-major tile in LDS (lds_pos layout, raw
// bf16 values; X0 = bf16(value inv)); the result replaces it. Every thread
// calls it, after a barrier that publishes the tile; it ends with one that
// publishes the result.
HM_DEV void ns_iterations(lds_u8* L, float inv, int steps, float ca, float cb, float cc, int round_once) {
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);  // wave-uniform: scalar branches
  u32x4_t x[KS];
  {
    const int ln = opaque_lane(lane);
    const int tr_krow = tr_krow_of(ln), tr_col = tr_col_of(ln);
#pragma unroll
    for (int k = 0; k < KS; ++k) x[k] = scale8_rne(col_frag(L, 32 * wave, k, tr_krow, tr_col), inv);
  }
  __syncthreads();  // every wave has its columns
#pragma unroll 1
  for (int it = 0; it < steps; ++it) {
    // ---- X by columns into LDS: row j of 256 holds column j of X -----------------
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
    with_part(wave, [&](auto part) {
      using P = decltype(part);
      u32x2_t o[5][4];
      gram_a<P>(L, lane, o);
      __syncthreads();  // every read of X is done
      gram_store<P>(L, lane, o);
      __syncthreads();
      gram_b<P>(L, lane, cb, cc, o);
      __syncthreads();  // every read of A is done
      gram_store<P>(L, lane, o);
    });
    __syncthreads();
    // ---- X' = bf16(bf16(B X) + a X) ------------------------------------------------
    u32x4_t o0[KS / 2], o1[KS / 2];
    apply_half<0>(L, lane, ca, round_once, x, o0, std::make_integer_sequence<int, KS>{});
    apply_half<4>(L, lane, ca, round_once, x, o1, std::make_integer_sequence<int, KS>{});
#pragma unroll
    for (int k = 0; k < KS / 2; ++k) {
      x[k] = o0[k];
      x[k + KS / 2] = o1[k];
    }
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
      for (int s = 0; s < 2; ++s) {
        const u32x2_t w = quad_transpose(u32x2_t{v[2 * s], v[2 * s + 1]}, kq);
        const int r = 16 * k + 8 * s + 4 * hi + kq;
        *reinterpret_cast<lds_u32x2*>(L + lds_pos(r, c >> 3, CH) + (c & 7) * 2) = w;
      }
    }
  }
  __syncthreads();
}

__global__ __launch_bounds__(NT, 1) void ns5_reg_kernel(const uint16_t* x, uint16_t* out,
                                                        const float* __restrict__ inv, int64_t ntiles, int steps,
                                                        float ca, float cb, float cc, int round_once) {
  __shared__ __attribute__((aligned(16))) uint8_t raw[LDS_BYTES];
  lds_u8* const L = (lds_u8*)raw;
  const int64_t t = blockIdx.x;  // one tile per workgroup
  if (t >= ntiles) return;
  const uint16_t* src = x + t * (int64_t)(T * T);
  uint16_t* dst = out + t * (int64_t)(T * T);
  const int tid = opaque_lane((int)threadIdx.x);
  u32x4_t v[T * CH / NT];
#pragma unroll
  for (int k = 0; k < T * CH / NT; ++k) v[k] = reinterpret_cast<const u32x4_t*>(src)[k * NT + tid];
  const float sc = inv[t];
#pragma unroll
  for (int k = 0; k < T * CH / NT; ++k) {
    const int idx = k * NT + tid;
    *reinterpret_cast<lds_u32x4*>(L + lds_pos(idx / CH, idx % CH, CH)) = v[k];
  }
  __syncthreads();
  ns_iterations(L, sc, steps, ca, cb, cc, round_once);
#pragma unroll
  for (int k = 0; k < T * CH / NT; ++k) {
    const int idx = k * NT + tid;
    reinterpret_cast<u32x4_t*>(dst)[idx] = *reinterpret_cast<lds_cu32x4*>(L + lds_pos(idx / CH, idx % CH, CH));
  }
}

// The normaliser of a tile from every wave's sum of squares of the two slabs it
// passed over (red[s][wave], published): slab 2 s + g is waves 4 g .. + 3 of
// pass s; the slabs in order, as tile_scale adds the gather's partials.
HM_DEV float tile_inv(const float (&red)[2][NT / 64], float eps) {
  float sum = 0.f;
  for (int q = 0; q < 4; ++q) {
    float p = 0.f;
    for (int i = 0; i < 4; ++i) p += red[q >> 1][4 * (q & 1) + i];
    sum += p;
  }
  return 1.0f / (sqrtf(sum) + eps);
}

// The whole optimizer step of a bucket of 256 x 256 NS tiles in one launch
// (tiles not transposed), as lds_step_kernel does it for 128 x 128: momentum
// and gather into LDS, the normaliser, the iterations, the untile with WD/LR.
// Per-element arithmetic and the order of the sum of squares are the separate
// kernels' (tile_step.h), so the step is bit-identical to gather ->
// tile_scale -> NS5 -> untile_apply. It saves the tile buffer's write and read
// and two reads of it by other launches; one workgroup fits a CU, so a tile's
// memory passes overlap only with the iterations of other CUs' tiles, which
// the one-tile-per-workgroup grid lets drift out of phase. Qwen3-0.6B set
// (6,720 tiles, bf16 parameters, fp32 grads): 3.53-3.54 ms a step against 4.24
// with the separate gather and untile launches; one 1024 x 1024 matrix (16
// tiles) 0.108 against 0.110 ms. 2 or 8 vectors in the gather's load batch and
// 4 in the untile's: within 0.6 %.
template <int DT, int PDT>
__global__ __launch_bounds__(NT, 1) void reg_step_kernel(const HimuonParamDesc* __restrict__ params, int n_params,
                                                         int64_t tile_begin, int64_t ntiles, int tile_h, int tile_w,
                                                         int steps, float ca, float cb, float cc, float eps,
                                                         int round_once, const float* __restrict__ sa) {
  __shared__ __attribute__((aligned(16))) uint8_t raw[LDS_BYTES];
  __shared__ float red[2][NT / 64];
  __shared__ float s_inv;
  lds_u8* const L = (lds_u8*)raw;
  const int64_t tt = blockIdx.x;
  if (tt >= ntiles) return;
#pragma unroll 1
  for (int s = 0; s < 2; ++s) {
    const float w = wave_sum(
        step_io<T, NT, DT, PDT, false, true, GAT_BATCH>(params, n_params, L, 0, tile_begin + tt, tile_h, tile_w, sa, s));
    if ((threadIdx.x & 63) == 0) red[s][threadIdx.x >> 6] = w;
  }
  __syncthreads();  // the tile and the waves' sums are in
  if (threadIdx.x == 0) s_inv = tile_inv(red, eps);
  __syncthreads();
  ns_iterations(L, s_inv, steps, ca, cb, cc, round_once);
#pragma unroll 1
  for (int s = 0; s < 2; ++s)
    step_io<T, NT, DT, PDT, true, false, UNT_BATCH>(params, n_params, L, tile_begin + tt, 0, tile_h, tile_w, sa, s);
}

// newton_schulz of a contiguous batch of plain matrices on 256 x 256 NS tiles in
// one launch, as ns_direct_lds_kernel (ns5_lds.hip) for 128 x 128.
template <int DT>
__global__ __launch_bounds__(NT, 1) void ns_direct_reg_kernel(const void* __restrict__ g, void* __restrict__ out,
                                                              int64_t ntiles, int rows, int cols, int steps, float ca,
                                                              float cb, float cc, float eps, int round_once) {
  __shared__ __attribute__((aligned(16))) uint8_t raw[LDS_BYTES];
  __shared__ float red[2][NT / 64];
  __shared__ float s_inv;
  lds_u8* const L = (lds_u8*)raw;
  const int64_t t = blockIdx.x;
  if (t >= ntiles) return;
#pragma unroll 1
  for (int s = 0; s < 2; ++s) {
    const float w = wave_sum(direct_load<T, NT, DT, 8>(g, L, t, rows, cols, s));
    if ((threadIdx.x & 63) == 0) red[s][threadIdx.x >> 6] = w;
  }
  __syncthreads();
  if (threadIdx.x == 0) s_inv = tile_inv(red, eps);
  __syncthreads();
  ns_iterations(L, s_inv, steps, ca, cb, cc, round_once);
#pragma unroll 1
  for (int s = 0; s < 2; ++s) direct_store<T, NT, DT>(out, L, t, rows, cols, s);
}

}  // namespace

void ns_direct_reg_run(const void* g, void* out, int64_t cnt, int rows, int cols, int dtype, int steps, float a,
                       float b, float c, float eps, bool round_once, hipStream_t s) {
  const auto run = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, dim3((unsigned)cnt), dim3(NT), 0, s, g, out, cnt, rows, cols, steps, a, b, c, eps,
                       round_once ? 1 : 0);
  };
  switch (dtype) {
    case HIMUON_DTYPE_F32: run(ns_direct_reg_kernel<HIMUON_DTYPE_F32>); break;
    case HIMUON_DTYPE_BF16: run(ns_direct_reg_kernel<HIMUON_DTYPE_BF16>); break;
    default: run(ns_direct_reg_kernel<HIMUON_DTYPE_F16>); break;
  }
}

bool reg_step_supported(int tile_h, int tile_w, int dtype, int param_dtype) {
  return tile_h > T / 2 && tile_h <= tile_w && tile_w <= T &&
         (dtype == HIMUON_DTYPE_F32 || dtype == HIMUON_DTYPE_BF16) &&
         (param_dtype == HIMUON_DTYPE_F32 || param_dtype == HIMUON_DTYPE_BF16);
}

void reg_step_run(const HimuonParamDesc* params, int n_params, int64_t tile_begin, int64_t cnt, int tile_h,
                  int tile_w, int dtype, int param_dtype, int steps, float a, float b, float c, float eps,
                  bool round_once, const float* sa, hipStream_t s) {
  for (int64_t off = 0; off < cnt; off += (int64_t)1 << 30) {
    const int64_t n = std::min<int64_t>(cnt - off, (int64_t)1 << 30);
    const auto run = [&](auto kernel) {
      hipLaunchKernelGGL(kernel, dim3((unsigned)n), dim3(NT), 0, s, params, n_params, tile_begin + off, n, tile_h,
                         tile_w, steps, a, b, c, eps, round_once ? 1 : 0, sa);
    };
    if (dtype == HIMUON_DTYPE_F32) {
      if (param_dtype == HIMUON_DTYPE_F32) run(reg_step_kernel<HIMUON_DTYPE_F32, HIMUON_DTYPE_F32>);
      else run(reg_step_kernel<HIMUON_DTYPE_F32, HIMUON_DTYPE_BF16>);
    } else {
      if (param_dtype == HIMUON_DTYPE_F32) run(reg_step_kernel<HIMUON_DTYPE_BF16, HIMUON_DTYPE_F32>);
      else run(reg_step_kernel<HIMUON_DTYPE_BF16, HIMUON_DTYPE_BF16>);
    }
  }
}

bool ns5_reg_supported(int mp, int np) { return mp == T && np == T; }

void ns5_reg_run(uint16_t* x, uint16_t* y, const float* inv, int64_t cnt, int steps, float a, float b, float c,
                 bool round_once, hipStream_t s) {
  uint16_t* out = (steps & 1) ? y : x;
  for (int64_t off = 0; off < cnt; off += (int64_t)1 << 30) {
    const int64_t n = std::min<int64_t>(cnt - off, (int64_t)1 << 30);
    hipLaunchKernelGGL(ns5_reg_kernel, dim3((unsigned)n), dim3(NT), 0, s, x + off * T * T, out + off * T * T,
                       inv + off, n, steps, a, b, c, round_once ? 1 : 0);
  }
}
