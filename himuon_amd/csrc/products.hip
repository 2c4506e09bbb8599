// The reference's three NS stage products for every operand dtype its kernels
// take: tl.dot on the loaded dtype with an fp32 accumulator, the result cast
// to the dtype of `out` (XXT.py:62-63, ba_plus_cAA.py:65-85,
// fused_bmm_add.py:73-88), tested there with bf16, fp16, fp32 and fp8 e5m2
// operands (tests/integration/test_kernels.py:36-165).
//
//   XXT          C = A A^T                     A: M x K       (mirrored store)
//   ba_plus_cAA  C = alpha A A^T + beta A      A: M x M       (mirrored store)
//   bmm_add      C = out(B X) + gamma X        B: M x M, X: M x N
//
// MFMA operands per input dtype (gfx950):
//   bf16          v_mfma_f32_32x32x16_bf16 on the values;
//   fp16          v_mfma_f32_32x32x16_f16 on the values;
//   fp8 e5m2      the same fp16 MFMA: an e5m2 byte is the upper byte of the
//                 fp16 with the same value (both have 5 exponent bits with
//                 bias 15), so widening is a shift and exact;
//   fp32          three bf16 MFMAs, hi*hi + hi*lo + lo*hi with hi = bf16(x)
//                 and lo = bf16(x - hi): 16 significant bits of every operand
//                 (TF32, which the reference's fp32 dot uses on its GPUs,
//                 keeps 11), each partial product exact in fp32.
// Output dtypes: fp32, bf16, fp16 (round to nearest even from fp32).
//
// The bf16-in / bf16-out products keep their own kernels (ns5_blk.hip,
// ns5_stream.hip), bit-identical to torch; these kernels serve every other
// dtype pair, and bf16 operands off 16-byte boundaries (ns_any_product: the same
// bits), which those kernels' direct-to-LDS loads do not take. Block tile 64 x 64
// x 64 or 128 x 128 x 64, four waves of one MFMA 32x32 tile each or of 2 x 2;
// operands are converted as they are staged through registers into a double
// buffer in LDS; the Gram products compute the lower blocks and store each block
// and its mirror.
//
// What bounds them: each K unit's loads, conversions and barrier in turn, so
// what counts is how many workgroups share a CU, until the operand stream of 64 x
// 64 blocks does (16-bit operands of long contractions: gram_128). us for XXT /
// ba_plus_cAA / bmm_add in fp32, 64 x 64 against 128 x 128 blocks: 8 of 512 x 1024
// 27 / 19 / 42 against 49 / 39 / 54 (59 / 49 / 55 with the mirrored block stored
// element by element and twice the instructions per conversion), 64 of 1024 x
// 2048 950 / 548 / 2370 against 1031 / 692 / 3121; fp16 8 of 512 x 1024 21 / 19 /
// 25 against 47 / 50 / 46.
#include <algorithm>

#include "ns5_kernels.h"

namespace {

constexpr int kThreads = 256;
constexpr int BK = 64;       // K per unit
constexpr int kAlign = 128;  // operand dimensions
constexpr int kLd = BK + 8;  // padded LDS row pitch (16-bit elements)

enum InType { kInF32 = HIMUON_DTYPE_F32, kInBf16 = HIMUON_DTYPE_BF16, kInF16 = HIMUON_DTYPE_F16,
              kInE5m2 = HIMUON_DTYPE_E5M2 };

typedef _Float16 f16x8_t __attribute__((ext_vector_type(8)));

template <int IN>
HM_DEV f32x16_t mfma_in(u32x4_t a, u32x4_t b, f32x16_t c) {
  if constexpr (IN == kInF16 || IN == kInE5m2)
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8_t, a), __builtin_bit_cast(f16x8_t, b),
                                                  c, 0, 0, 0);
  else
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8_t, a),
                                                   __builtin_bit_cast(bf16x8_t, b), c, 0, 0, 0);
}

// 8 consecutive input elements as 16-bit MFMA operands: `hi` always, `lo`
// (the fp32 remainder) for fp32 inputs. (fp32 and 16-bit operands at any element
// alignment, as load8.)
struct Oct {
  u32x4_t hi, lo;
};

HM_DEV uint32_t e5m2_pair(uint32_t w, int k) {  // bytes 2k, 2k+1 of w -> two fp16
  const uint32_t b0 = (w >> (16 * k)) & 0xffu, b1 = (w >> (16 * k + 8)) & 0xffu;
  return (b0 << 8) | (b1 << 24);
}

template <int IN>
HM_DEV Oct load_oct(const void* base, int64_t idx) {
  Oct o;
  if constexpr (IN == kInF32) {
    const float* p = static_cast<const float*>(base) + idx;
    const f32x4_any v0 = *reinterpret_cast<const f32x4_any*>(p);
    const f32x4_any v1 = *reinterpret_cast<const f32x4_any*>(p + 4);
    float x[8] = {v0[0], v0[1], v0[2], v0[3], v1[0], v1[1], v1[2], v1[3]};
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      o.hi[k] = pk_bf16(x[2 * k], x[2 * k + 1]);
      const float h0 = __uint_as_float(o.hi[k] << 16), h1 = __uint_as_float(o.hi[k] & 0xffff0000u);
      // (an infinite or NaN hi carries the value alone)
      o.lo[k] = pk_bf16(__builtin_isfinite(h0) ? x[2 * k] - h0 : 0.f, __builtin_isfinite(h1) ? x[2 * k + 1] - h1 : 0.f);
    }
  } else if constexpr (IN == kInE5m2) {
    const u32x2_t w = *reinterpret_cast<const u32x2_t*>(static_cast<const uint8_t*>(base) + idx);
    o.hi = u32x4_t{e5m2_pair(w[0], 0), e5m2_pair(w[0], 1), e5m2_pair(w[1], 0), e5m2_pair(w[1], 1)};
    o.lo = u32x4_t{0u, 0u, 0u, 0u};
  } else {
    o.hi = *reinterpret_cast<const u32x4_any*>(static_cast<const uint16_t*>(base) + idx);
    o.lo = u32x4_t{0u, 0u, 0u, 0u};
  }
  return o;
}

template <int IN>
HM_DEV float load_elem_in(const void* base, int64_t idx) {
  if constexpr (IN == kInF32) return static_cast<const float*>(base)[idx];
  else if constexpr (IN == kInBf16) return bf16_to_f32(static_cast<const uint16_t*>(base)[idx]);
  else if constexpr (IN == kInF16) return f16_to_f32(static_cast<const uint16_t*>(base)[idx]);
  else return f16_to_f32((uint16_t)(static_cast<const uint8_t*>(base)[idx] << 8));
}

HM_DEV float round_out(float v, int out_dtype) {
  if (out_dtype == HIMUON_DTYPE_BF16) return round_bf16(v);
  if (out_dtype == HIMUON_DTYPE_F16) return f16_to_f32(f32_to_f16(v));
  return v;
}

HM_DEV void store_out(void* base, int64_t idx, float v, int out_dtype) {
  if (out_dtype == HIMUON_DTYPE_F32)
    static_cast<float*>(base)[idx] = v;
  else if (out_dtype == HIMUON_DTYPE_BF16)
    static_cast<uint16_t*>(base)[idx] = (uint16_t)f32_to_bf16(v);
  else
    static_cast<uint16_t*>(base)[idx] = f32_to_f16(v);
}

constexpr int planes(int in) { return in == kInF32 ? 2 : 1; }

// acc += a b of one MFMA tile and k-step (fp32 operands: lo hi, hi lo, hi hi).
template <int IN>
HM_DEV void product(const u32x4_t (&a)[planes(IN)], const u32x4_t (&b)[planes(IN)], f32x16_t& acc) {
  if constexpr (planes(IN) == 2) {
    acc = mfma_in<IN>(a[1], b[0], acc);
    acc = mfma_in<IN>(a[0], b[1], acc);
  }
  acc = mfma_in<IN>(a[0], b[0], acc);
}

// 4 consecutive outputs, at any element alignment.
HM_DEV void store_out4(void* base, int64_t idx, const float (&v)[4], int out_dtype) {
  if (out_dtype == HIMUON_DTYPE_F32) {
    *reinterpret_cast<f32x4_any*>(static_cast<float*>(base) + idx) = f32x4_any{v[0], v[1], v[2], v[3]};
  } else {
    typedef uint32_t u32x2_any __attribute__((ext_vector_type(2), aligned(2)));
    u32x2_any w;
    if (out_dtype == HIMUON_DTYPE_BF16)
      w = u32x2_any{pack2(f32_to_bf16(v[0]), f32_to_bf16(v[1])), pack2(f32_to_bf16(v[2]), f32_to_bf16(v[3]))};
    else
      w = u32x2_any{pack2(f32_to_f16(v[0]), f32_to_f16(v[1])), pack2(f32_to_f16(v[2]), f32_to_f16(v[3]))};
    *reinterpret_cast<u32x2_any*>(static_cast<uint16_t*>(base) + idx) = w;
  }
}

// C = alpha S S^T (+ beta S when add_s; K == M) for each batch entry; S:
// M x K, C: M x M. Lower BT x BT blocks only, each stored at (bi, bj) and
// mirrored (a lane holds 4 consecutive rows of a column: 4 consecutive
// elements of the mirrored row). BT: the block's edge, 64 or 128.
template <int IN, int BT>
__global__ __launch_bounds__(kThreads) void prod_gram_kernel(const void* __restrict__ S, void* __restrict__ C,
                                                             int M, int K, int64_t first, int64_t count,
                                                             float alpha, float beta, int add_s, int out_dtype) {
  constexpr int NP = planes(IN);
  constexpr int R = BT / 32;   // loader rows per thread
  constexpr int WT = BT / 64;  // MFMA tiles per wave and direction
  __shared__ __attribute__((aligned(16))) uint16_t sI[2][NP][BT * kLd];
  __shared__ __attribute__((aligned(16))) uint16_t sJ[2][NP][BT * kLd];

  const int nb = M / BT;
  const int npairs = nb * (nb + 1) / 2;
  const int64_t local = xcd_item(count);
  if (local >= count) return;
  const int64_t item = first + local;
  const int64_t tile = item / npairs;
  const int p = (int)(item % npairs);
  int bi = 0;
  while ((bi + 1) * (bi + 2) / 2 <= p) ++bi;
  const int bj = p - bi * (bi + 1) / 2;

  const int64_t s0 = tile * (int64_t)M * K;  // element index of the tile
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int wm = wave >> 1, wn = wave & 1;
  const int lrow = tid >> 3, lkv = (tid & 7) * 8;  // loader: rows lrow + 32q, k offset lkv

  Oct ra[R], rb[R];
  auto gload = [&](int k0) {
#pragma unroll
    for (int q = 0; q < R; ++q) {
      const int row = lrow + 32 * q;
      ra[q] = load_oct<IN>(S, s0 + (int64_t)(bi * BT + row) * K + k0 + lkv);
      rb[q] = load_oct<IN>(S, s0 + (int64_t)(bj * BT + row) * K + k0 + lkv);
    }
  };
  auto lstore = [&](int buf) {
#pragma unroll
    for (int q = 0; q < R; ++q) {
      const int row = lrow + 32 * q;
      *reinterpret_cast<u32x4_t*>(&sI[buf][0][row * kLd + lkv]) = ra[q].hi;
      *reinterpret_cast<u32x4_t*>(&sJ[buf][0][row * kLd + lkv]) = rb[q].hi;
      if constexpr (NP == 2) {
        *reinterpret_cast<u32x4_t*>(&sI[buf][NP - 1][row * kLd + lkv]) = ra[q].lo;
        *reinterpret_cast<u32x4_t*>(&sJ[buf][NP - 1][row * kLd + lkv]) = rb[q].lo;
      }
    }
  };

  f32x16_t acc[WT][WT];
#pragma unroll
  for (int mi = 0; mi < WT; ++mi)
#pragma unroll
    for (int ni = 0; ni < WT; ++ni)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[mi][ni][r] = 0.f;

  const int nk = K / BK;
  gload(0);
  lstore(0);
  __syncthreads();
  for (int kt = 0; kt < nk; ++kt) {
    const int cur = kt & 1;
    if (kt + 1 < nk) gload((kt + 1) * BK);
#pragma unroll
    for (int ks = 0; ks < BK / 16; ++ks) {
      const int kk = ks * 16 + (lane >> 5) * 8;
      u32x4_t a[WT][NP], b[WT][NP];
#pragma unroll
      for (int t = 0; t < WT; ++t)
#pragma unroll
        for (int pl = 0; pl < NP; ++pl) {
          a[t][pl] = *reinterpret_cast<const u32x4_t*>(&sI[cur][pl][(wm * 32 * WT + 32 * t + (lane & 31)) * kLd + kk]);
          b[t][pl] = *reinterpret_cast<const u32x4_t*>(&sJ[cur][pl][(wn * 32 * WT + 32 * t + (lane & 31)) * kLd + kk]);
        }
#pragma unroll
      for (int mi = 0; mi < WT; ++mi)
#pragma unroll
        for (int ni = 0; ni < WT; ++ni) product<IN>(a[mi], b[ni], acc[mi][ni]);
    }
    if (kt + 1 < nk) lstore(cur ^ 1);
    __syncthreads();
  }

  // MFMA 32x32 output layout: register r of lane l holds row
  // 8 (r / 4) + 4 (l / 32) + r % 4, column l % 32.
  const int64_t c0 = tile * (int64_t)M * M;
  const bool offdiag = bi > bj;
#pragma unroll
  for (int mi = 0; mi < WT; ++mi)
#pragma unroll
    for (int ni = 0; ni < WT; ++ni)
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int i0 = bi * BT + wm * 32 * WT + 32 * mi + 8 * q + 4 * (lane >> 5);
        const int j = bj * BT + wn * 32 * WT + 32 * ni + (lane & 31);
        float v[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          v[e] = alpha * acc[mi][ni][4 * q + e];
          if (add_s) v[e] = fmaf(beta, load_elem_in<IN>(S, s0 + (int64_t)(i0 + e) * K + j), v[e]);
          if (offdiag || i0 + e >= j) store_out(C, c0 + (int64_t)(i0 + e) * M + j, v[e], out_dtype);
        }
        if (offdiag || i0 > j) {  // all 4 below the diagonal
          store_out4(C, c0 + (int64_t)j * M + i0, v, out_dtype);
        } else {
#pragma unroll
          for (int e = 0; e < 4; ++e)
            if (i0 + e > j) store_out(C, c0 + (int64_t)j * M + i0 + e, v[e], out_dtype);
        }
      }
}

// C = out(Bm X) + gamma X for each batch entry (Bm X rounded to the output
// dtype before the add, fused_bmm_add.py:73-88, unless ONCE); Bm: M x M, X and
// C: M x N.
// X is the MFMA B operand with the contraction along its rows: each 4 x 8
// block of X is transposed into the k-octet-major LDS layout sX[k/8][j][k%8].
template <int IN, int BT, bool ONCE>
__global__ __launch_bounds__(kThreads) void prod_apply_kernel(const void* __restrict__ Bm,
                                                              const void* __restrict__ X, void* __restrict__ C,
                                                              int M, int N, int64_t first, int64_t count,
                                                              float gamma, int out_dtype) {
  constexpr int NP = planes(IN);
  constexpr int R = BT / 32;   // loader rows per thread
  constexpr int WT = BT / 64;  // MFMA tiles per wave and direction
  __shared__ __attribute__((aligned(16))) uint16_t sA[2][NP][BT * kLd];
  __shared__ __attribute__((aligned(16))) uint16_t sX[2][NP][(BK / 8) * BT * 8];

  const int nbi = M / BT, nbj = N / BT;
  const int blocks = nbi * nbj;
  const int64_t local = xcd_item(count);
  if (local >= count) return;
  const int64_t item = first + local;
  const int64_t tile = item / blocks;
  const int blk = (int)(item % blocks);
  const int bi = blk / nbj, bj = blk % nbj;

  const int64_t b0 = tile * (int64_t)M * M, x0 = tile * (int64_t)M * N;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int wm = wave >> 1, wn = wave & 1;
  const int lrow = tid >> 3, lkv = (tid & 7) * 8;  // Bm loader
  const int xk = tid / (BT / 8) * R, xjo = tid % (BT / 8) * 8;  // X loader: rows xk .. + R - 1, columns xjo .. + 7

  Oct ra[R], rx[R];
  auto gload = [&](int k0) {
#pragma unroll
    for (int q = 0; q < R; ++q) {
      const int row = lrow + 32 * q;
      ra[q] = load_oct<IN>(Bm, b0 + (int64_t)(bi * BT + row) * M + k0 + lkv);
    }
#pragma unroll
    for (int rr = 0; rr < R; ++rr) rx[rr] = load_oct<IN>(X, x0 + (int64_t)(k0 + xk + rr) * N + bj * BT + xjo);
  };
  auto lstore = [&](int buf) {
#pragma unroll
    for (int q = 0; q < R; ++q) {
      const int row = lrow + 32 * q;
      *reinterpret_cast<u32x4_t*>(&sA[buf][0][row * kLd + lkv]) = ra[q].hi;
      if constexpr (NP == 2) *reinterpret_cast<u32x4_t*>(&sA[buf][NP - 1][row * kLd + lkv]) = ra[q].lo;
    }
#pragma unroll
    for (int pl = 0; pl < NP; ++pl) {
      uint16_t* base = &sX[buf][pl][(xk >> 3) * BT * 8 + (xk & 7)];
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const int w = e >> 1, h = e & 1;
        auto v = [&](int rr) { return half16(pl == 0 ? rx[rr].hi[w] : rx[rr].lo[w], h); };
#pragma unroll
        for (int rr = 0; rr < R; rr += 2)
          *reinterpret_cast<uint32_t*>(base + (xjo + e) * 8 + rr) = pack2(v(rr), v(rr + 1));
      }
    }
  };

  f32x16_t acc[WT][WT];
#pragma unroll
  for (int mi = 0; mi < WT; ++mi)
#pragma unroll
    for (int ni = 0; ni < WT; ++ni)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[mi][ni][r] = 0.f;

  const int nk = M / BK;
  gload(0);
  lstore(0);
  __syncthreads();
  for (int kt = 0; kt < nk; ++kt) {
    const int cur = kt & 1;
    if (kt + 1 < nk) gload((kt + 1) * BK);
#pragma unroll
    for (int ks = 0; ks < BK / 16; ++ks) {
      const int kk = ks * 16 + (lane >> 5) * 8;
      const int koct = ks * 2 + (lane >> 5);
      u32x4_t a[WT][NP], b[WT][NP];
#pragma unroll
      for (int t = 0; t < WT; ++t)
#pragma unroll
        for (int pl = 0; pl < NP; ++pl) {
          a[t][pl] = *reinterpret_cast<const u32x4_t*>(&sA[cur][pl][(wm * 32 * WT + 32 * t + (lane & 31)) * kLd + kk]);
          b[t][pl] =
              *reinterpret_cast<const u32x4_t*>(&sX[cur][pl][(koct * BT + wn * 32 * WT + 32 * t + (lane & 31)) * 8]);
        }
#pragma unroll
      for (int mi = 0; mi < WT; ++mi)
#pragma unroll
        for (int ni = 0; ni < WT; ++ni) product<IN>(a[mi], b[ni], acc[mi][ni]);
    }
    if (kt + 1 < nk) lstore(cur ^ 1);
    __syncthreads();
  }

#pragma unroll
  for (int mi = 0; mi < WT; ++mi)
#pragma unroll
    for (int ni = 0; ni < WT; ++ni)
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int i = bi * BT + wm * 32 * WT + 32 * mi + 8 * (r >> 2) + 4 * (lane >> 5) + (r & 3);
        const int j = bj * BT + wn * 32 * WT + 32 * ni + (lane & 31);
        const int64_t e = x0 + (int64_t)i * N + j;
        const float bx = ONCE ? acc[mi][ni][r] : round_out(acc[mi][ni][r], out_dtype);
        store_out(C, e, bx + gamma * load_elem_in<IN>(X, e), out_dtype);
      }
}

bool dtype_in_ok(int d) {
  return d == HIMUON_DTYPE_F32 || d == HIMUON_DTYPE_BF16 || d == HIMUON_DTYPE_F16 || d == HIMUON_DTYPE_E5M2;
}
bool dtype_out_ok(int d) { return d == HIMUON_DTYPE_F32 || d == HIMUON_DTYPE_BF16 || d == HIMUON_DTYPE_F16; }

// Launches of at most 2^23 work items: a grid holds fewer than 2^32 threads,
// which a result near the size of the memory exceeds in 64 x 64 blocks.
constexpr int64_t kLaunchItems = int64_t(1) << 23;

template <int IN, int BT>
void launch_gram_blocks(const void* s, void* c, int M, int K, int64_t batch, float alpha, float beta, int add_s, int od,
                        hipStream_t st) {
  const int64_t nb = M / BT, items = batch * (nb * (nb + 1) / 2);
  for (int64_t first = 0; first < items; first += kLaunchItems) {
    const int64_t count = std::min(kLaunchItems, items - first);
    hipLaunchKernelGGL((prod_gram_kernel<IN, BT>), dim3((unsigned)xcd_grid(count)), dim3(kThreads), 0, st, s, c, M, K, first,
                       count, alpha, beta, add_s, od);
  }
}

template <int IN, int BT, bool ONCE>
void launch_apply_blocks(const void* b, const void* x, void* c, int M, int N, int64_t batch, float gamma, int od,
                         hipStream_t st) {
  const int64_t items = batch * (M / BT) * (N / BT);
  for (int64_t first = 0; first < items; first += kLaunchItems) {
    const int64_t count = std::min(kLaunchItems, items - first);
    hipLaunchKernelGGL((prod_apply_kernel<IN, BT, ONCE>), dim3((unsigned)xcd_grid(count)), dim3(kThreads), 0, st, b, x, c, M, N,
                       first, count, gamma, od);
  }
}

// 128 x 128 blocks where 64 x 64 ones, which stream each operand twice as often,
// would be bound by that: long contractions of many blocks. `items`: 128 x 128
// blocks, K: the contraction. The lines lie between shapes measured both ways (us,
// 64 x 64 / 128 x 128; MxK the operand of XXT, a square one that of ba_plus_cAA):
//   Gram, 16-bit to fp32, K >= 1024 and items K >= 2^21: 64 of 1024 x 1024 214 / 178,
//     8 of 2048 x 2048 132 / 123, 4096 x 4096 167 / 132, 8192 x 8192 1267 / 748; below
//     it 4 of 2048 x 2048 83 / 102, 16 of 1024 x 1024 52 / 75.
//   Gram, 16-bit to 16-bit (dearer stores), K >= 4096 and items K >= 3.5 2^20: 3072 x
//     12288 277 / 215, 64 of 1024 x 4096 593 / 489, 8192 x 8192 1254 / 802, below it
//     8 of 2048 x 2048 150 / 170; and from 6144 rows on, 6144 x 2048 203 / 177.
//   Gram, e5m2 (half the bytes), K >= 4096 and items K >= 7 2^20: 4 of 4096 x 4096
//     541 / 516, 8192 x 8192 1050 / 893, below it 2 of 4096 x 4096 278 / 313.
//   Apply, 16-bit to fp32, M >= 2048 and items M >= 2^22: 8 of 2048 x 2048 385 / 361,
//     8192 x 8192 2773 / 2568, below it 64 of 1024 x 1024 407 / 438.
//   Apply, 16-bit to 16-bit, M >= 4096 and items M >= 2^23: 4 of 4096 x 2048 758 /
//     703, 8192 x 8192 2786 / 2637, below it 4096 x 4096 370 / 376.
//   Apply of e5m2 and every product of fp32 operands: 64 x 64 throughout.
template <int IN>
bool gram_128(int64_t items, int M, int K, int od) {
  const int64_t work = items * K;
  if (IN == kInE5m2) return K >= 4096 && work >= 7 << 20;
  if (od == HIMUON_DTYPE_F32) return K >= 1024 && work >= 1 << 21;
  return (K >= 4096 && work >= 7 << 19) || (M >= 6144 && K >= 1024);
}

bool apply_128(int64_t items, int M, int od) {
  return od == HIMUON_DTYPE_F32 ? M >= 2048 && items * M >= 1 << 22 : M >= 4096 && items * M >= 1 << 23;
}

template <int IN>
void launch_gram(const void* s, void* c, int M, int K, int64_t batch, float alpha, float beta, int add_s, int od,
                 hipStream_t st) {
  if constexpr (IN != kInF32) {
    const int64_t nb = M / 128;
    if (gram_128<IN>(batch * (nb * (nb + 1) / 2), M, K, od))
      return launch_gram_blocks<IN, 128>(s, c, M, K, batch, alpha, beta, add_s, od, st);
  }
  launch_gram_blocks<IN, 64>(s, c, M, K, batch, alpha, beta, add_s, od, st);
}

template <int IN, bool ONCE = false>
void launch_apply(const void* b, const void* x, void* c, int M, int N, int64_t batch, float gamma, int od,
                  hipStream_t st) {
  if constexpr (IN != kInF32 && IN != kInE5m2) {
    if (apply_128(batch * (M / 128) * (N / 128), M, od))
      return launch_apply_blocks<IN, 128, ONCE>(b, x, c, M, N, batch, gamma, od, st);
  }
  launch_apply_blocks<IN, 64, ONCE>(b, x, c, M, N, batch, gamma, od, st);
}

// 128 x 128 output blocks a call takes.
constexpr int64_t kMaxItems = (int64_t(1) << 31) - 8;

int gram(const void* s, void* c, int M, int K, int64_t batch, float alpha, float beta, int add_s, int id, int od,
         void* stream) {
  if (!s || !c || s == c || batch < 0 || M <= 0 || K <= 0 || M % kAlign || K % BK || !dtype_in_ok(id) ||
      !dtype_out_ok(od) || (add_s && K != M))
    return HIMUON_EINVAL;
  if (batch == 0) return 0;
  const int64_t nb = M / kAlign;
  if (batch > kMaxItems / (nb * (nb + 1) / 2)) return HIMUON_EINVAL;
  const hipStream_t st = static_cast<hipStream_t>(stream);
  switch (id) {
    case HIMUON_DTYPE_F32: launch_gram<kInF32>(s, c, M, K, batch, alpha, beta, add_s, od, st); break;
    case HIMUON_DTYPE_BF16: launch_gram<kInBf16>(s, c, M, K, batch, alpha, beta, add_s, od, st); break;
    case HIMUON_DTYPE_F16: launch_gram<kInF16>(s, c, M, K, batch, alpha, beta, add_s, od, st); break;
    default: launch_gram<kInE5m2>(s, c, M, K, batch, alpha, beta, add_s, od, st); break;
  }
  return (int)hipGetLastError();
}

}  // namespace

void ns_any_product(int mode, const NsProduct& g, hipStream_t s) {
  if (mode == kApply && g.round_once)
    launch_apply<kInBf16, true>(g.P, g.Q, g.C, g.M, g.N, g.ntiles, g.beta, HIMUON_DTYPE_BF16, s);
  else if (mode == kApply)
    launch_apply<kInBf16>(g.P, g.Q, g.C, g.M, g.N, g.ntiles, g.beta, HIMUON_DTYPE_BF16, s);
  else
    launch_gram<kInBf16>(g.P, g.C, g.M, g.K, g.ntiles, g.alpha, g.beta, mode == kGramB, HIMUON_DTYPE_BF16, s);
}

extern "C" int himuon_xxt_typed(const void* x, void* out, int64_t batch, int M, int K, int in_dtype,
                                int out_dtype, void* stream) {
  return gram(x, out, M, K, batch, 1.f, 0.f, 0, in_dtype, out_dtype, stream);
}

extern "C" int himuon_ba_plus_caa_typed(const void* a, void* out, int64_t batch, int M, float alpha, float beta,
                                        int in_dtype, int out_dtype, void* stream) {
  return gram(a, out, M, M, batch, alpha, beta, 1, in_dtype, out_dtype, stream);
}

extern "C" int himuon_bmm_add_typed(const void* b, const void* x, void* out, int64_t batch, int M, int N, float a,
                                    int in_dtype, int out_dtype, void* stream) {
  if (!b || !x || !out || out == x || out == b || batch < 0 || M <= 0 || N <= 0 || M % kAlign || N % kAlign ||
      !dtype_in_ok(in_dtype) || !dtype_out_ok(out_dtype))
    return HIMUON_EINVAL;
  if (batch == 0) return 0;
  const int64_t blocks = (int64_t)(M / kAlign) * (N / kAlign);
  if (batch > kMaxItems / blocks) return HIMUON_EINVAL;
  const hipStream_t st = static_cast<hipStream_t>(stream);
  switch (in_dtype) {
    case HIMUON_DTYPE_F32: launch_apply<kInF32>(b, x, out, M, N, batch, a, out_dtype, st); break;
    case HIMUON_DTYPE_BF16: launch_apply<kInBf16>(b, x, out, M, N, batch, a, out_dtype, st); break;
    case HIMUON_DTYPE_F16: launch_apply<kInF16>(b, x, out, M, N, batch, a, out_dtype, st); break;
    default: launch_apply<kInE5m2>(b, x, out, M, N, batch, a, out_dtype, st); break;
  }
  return (int)hipGetLastError();
}
