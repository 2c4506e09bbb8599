// Batched quintic Newton-Schulz (NS5) on gfx950 bf16 MFMA, fp32 accumulation.
//
// Per NS tile (m x n, m <= n, zero padded to mp x np) and per iteration:
//   A = bf16(X X^T)
//   B = bf16(c A A^T + b A)
//   X = bf16(bf16(B X) + a X)
// following the rounding points of the reference kernels
// (triton_kernels/XXT.py:55-75, ba_plus_cAA.py:58-85, fused_bmm_add.py:65-88,
// ns5_smem.py:84-101). A and B are symmetric: only their lower-triangular
// blocks are computed, each stored twice (as itself and mirrored).
//
// Iteration 0 reads the raw bf16 tile and applies the per-tile Frobenius
// normaliser as the operands enter: X0 = bf16(x * inv[t])
// (himuon.py:242, ns5_smem.py:84-87).
//
// This file holds the C entry points and the choice of kernels for a geometry.
#include <algorithm>
#include <atomic>
#include <mutex>

#include "ns5_kernels.h"

namespace {

constexpr int kThreads = 256;
constexpr int BM = 128;  // edges are multiples of this
constexpr int kScaleRows = 768;  // padded rows from which X0 is written first

// X = bf16(X inv[t]) in place: the result of steps == 0, and X0 of matrices
// whose products would otherwise scale each value many times (ns5_impl). A
// workgroup covers kScaleVec 16-byte vectors per thread of one tile.
constexpr int kScaleVec = 8;
__global__ __launch_bounds__(kThreads) void ns_scale_kernel(uint16_t* __restrict__ X, const float* __restrict__ inv,
                                                            int64_t vec_per_tile, int64_t wgs_per_tile) {
  const int64_t t = blockIdx.x / wgs_per_tile;
  const int64_t v0 = (blockIdx.x - t * wgs_per_tile) * (kThreads * kScaleVec) + threadIdx.x;
  u32x4_any* const x = reinterpret_cast<u32x4_any*>(X) + t * vec_per_tile;  // (any alignment, as load8)
  const float s = inv[t];
  u32x4_t v[kScaleVec];
#pragma unroll
  for (int k = 0; k < kScaleVec; ++k)
    if (v0 + k * kThreads < vec_per_tile) v[k] = x[v0 + k * kThreads];
#pragma unroll
  for (int k = 0; k < kScaleVec; ++k)
    if (v0 + k * kThreads < vec_per_tile) x[v0 + k * kThreads] = scale8(v[k], s);
}

void ns_scale(uint16_t* x, const float* inv, int64_t n_tiles, int64_t rect, hipStream_t s) {
  const int64_t vpt = rect / 8, wgs = (vpt + kThreads * kScaleVec - 1) / (kThreads * kScaleVec);
  const int64_t most = std::max<int64_t>(1, launch_wgs(kThreads) / wgs);  // tiles per launch
  for (int64_t t = 0; t < n_tiles; t += most)
    hipLaunchKernelGGL(ns_scale_kernel, dim3((unsigned)(std::min(most, n_tiles - t) * wgs)), dim3(kThreads), 0, s,
                       x + t * rect, inv + t, vpt, wgs);
}

}  // namespace

extern "C" size_t himuon_ns5_workspace_bytes(int64_t sub_batch, int mp, int np) {
  if (sub_batch <= 0 || mp <= 0 || np <= 0) return 0;
  return 2 * (size_t)sub_batch * mp * mp * sizeof(uint16_t);  // A and B per sub-batch tile
}

namespace {
// himuon_ns5_ex, and with `untile` (himuon_ns5_untile_apply; the caller has
// checked that the fused path applies) the untile with WD/LR fused into the
// last iteration: its tile0 is the bucket index of tile 0 of x.
int ns5_impl(uint16_t* x, uint16_t* y, const float* inv, int64_t n_tiles, int mp, int np, int steps, float a,
             float b, float c, void* workspace, size_t workspace_bytes, int64_t sub_batch, int flags,
             void* stream, const BaUntile* untile) {
  const int family = flags & HIMUON_NS_FAMILY_MASK;
  const bool round_once = (flags & HIMUON_NS_ROUND_ONCE) != 0;
  const int rows = (flags & HIMUON_NS_ROWS_MASK) >> HIMUON_NS_ROWS_SHIFT;
  if (!x || !y || x == y || !inv || n_tiles < 0 || steps < 0 || mp <= 0 || np <= 0 || mp > np ||
      mp % HIMUON_NS_ALIGN || np % HIMUON_NS_ALIGN || sub_batch <= 0 || rows > 64 ||
      (flags & ~(HIMUON_NS_FAMILY_MASK | HIMUON_NS_ROUND_ONCE | HIMUON_NS_ROWS_MASK)) ||
      (family != HIMUON_NS_FAMILY_AUTO && family != HIMUON_NS_FAMILY_BLOCK128 &&
       family != HIMUON_NS_FAMILY_STREAM3))
    return HIMUON_EINVAL;
  if (n_tiles == 0) return 0;
  const int64_t sb = sub_batch < n_tiles ? sub_batch : n_tiles;
  if (steps > 0 && (!workspace || workspace_bytes < himuon_ns5_workspace_bytes(sb, mp, np)))
    return HIMUON_ENOSPC;
  const hipStream_t s = static_cast<hipStream_t>(stream);
  const int64_t sq = (int64_t)mp * mp, rect = (int64_t)mp * np;

  if (steps == 0) {  // X0 = bf16(x * inv), in place (the result of an even step count is in x)
    ns_scale(x, inv, n_tiles, rect, s);
    return (int)hipGetLastError();
  }

  uint16_t* wsA = static_cast<uint16_t*>(workspace);
  uint16_t* wsB = wsA + sb * sq;
  // Family AUTO: tiles whose padded edges are multiples of 256 run three
  // products per iteration, each on the faster block size (ns_product); tiles with mp == 128
  // and np in {128, 256, 512} run the fused LDS-resident kernel (ns5_lds.hip),
  // 256 x 256 tiles the one that keeps X in registers (ns5_reg.hip: 16 tiles
  // 0.086 against 0.187 ms for the streamed products, 256 tiles 0.105 against
  // 0.34, 6,720 tiles 2.45-2.55 against 6.13-6.25 ms, same box); other tiles
  // run the 128-block kernels (ns5_blk.hip), which family BLOCK128 selects for every
  // geometry.
  // 512 x 512 tiles run the other two products fused (ns5_ba.hip); family
  // STREAM3 runs three products on 256 x 256 blocks.
  const bool small = family == HIMUON_NS_FAMILY_BLOCK128;
  const bool few_rows = family == HIMUON_NS_FAMILY_AUTO && ns5_small_supported(rows, mp, np);
  const bool st = ns5_stream_supported(mp, np) && !small;
  const bool lds = ns5_lds_supported(mp, np) && !small;
  // (buffers off 16-byte boundaries: ns_any_product on X0, no fused pair)
  const bool aligned = dma_aligned(x, y, workspace);
  const bool ba = ns5_ba_supported(mp, np) && family == HIMUON_NS_FAMILY_AUTO && (aligned || untile);
  const bool reg = ns5_reg_supported(mp, np) && family == HIMUON_NS_FAMILY_AUTO;

  // Matrices of many blocks: the products of the first iteration would scale
  // every X value once per block that reads it (9 times in GramA and 8 in Apply
  // at 1024 rows), beside MFMAs that leave no time for it; X0 is written in its
  // place once instead. Five iterations of 56 matrices of 1024 x 3072 3.78-3.83
  // against 3.91-3.95 ms, of 12 of 896 x 2432 0.66-0.67 against 0.68-0.69, of 60
  // of 768 x 768 0.92-0.93 against 0.93-0.94; from 512 rows on, 400 of 512 x 768
  // would be slower (2.65 against 2.56-2.60 ms).
  const bool scale_first = !few_rows && !lds && !reg &&
                           ((family == HIMUON_NS_FAMILY_AUTO && mp >= kScaleRows) || !aligned);
  for (int64_t s0 = 0; s0 < n_tiles; s0 += sb) {
    const int64_t cnt = std::min<int64_t>(sb, n_tiles - s0);
    const int64_t o = s0 * rect;
    if (scale_first) ns_scale(x + o, inv + s0, cnt, rect, s);
    const float* const first_inv = scale_first ? nullptr : inv + s0;
    if (few_rows) {
      if (!ns5_small_run(x + o, y + o, inv + s0, cnt, rows, np, steps, a, b, c, round_once, s)) return HIMUON_EINVAL;
    } else if (lds) {
      ns5_lds_run(x + o, y + o, inv + s0, cnt, mp, np, steps, a, b, c, round_once, s);
    } else if (reg) {
      ns5_reg_run(x + o, y + o, inv + s0, cnt, steps, a, b, c, round_once, s);
    } else if (st) {
      BaUntile u{};
      if (untile) {
        u = *untile;
        u.tile0 += s0;
      }
      const int rc = ns5_stream_run(x + o, y + o, first_inv, cnt, mp, np, steps, a, b, c, round_once, ba,
                                    family == HIMUON_NS_FAMILY_AUTO, wsA, wsB, s, untile ? &u : nullptr);
      if (rc) return rc;
    } else {
      const uint16_t* cur = x + o;
      uint16_t* nxt = y + o;
      const float* cur_inv = first_inv;
      for (int it = 0; it < steps; ++it) {
        ns_blk_product(kGramA, NsProduct{cur, rect, np, cur, rect, np, nullptr, 0, 0, wsA, sq, mp, mp, mp, np, cnt, 1.f, 0.f,
                                  0, cur_inv}, s);
        ns_blk_product(kGramB, NsProduct{wsA, sq, mp, wsA, sq, mp, wsA, sq, mp, wsB, sq, mp, mp, mp, mp, cnt, c, b, 0,
                                  nullptr}, s);
        ns_blk_product(kApply, NsProduct{wsB, sq, mp, cur, rect, np, cur, rect, np, nxt, rect, np, mp, np, mp, cnt, 1.f, a,
                                  round_once ? 1 : 0, cur_inv}, s);
        const uint16_t* t = cur;
        cur = nxt;
        nxt = const_cast<uint16_t*>(t);
        cur_inv = nullptr;
      }
    }
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return (int)e;
  }
  return 0;
}
}  // namespace

extern "C" int himuon_ns5_ex(uint16_t* x, uint16_t* y, const float* inv, int64_t n_tiles, int mp,
                             int np, int steps, float a, float b, float c, void* workspace,
                             size_t workspace_bytes, int64_t sub_batch, int flags, void* stream) {
  return ns5_impl(x, y, inv, n_tiles, mp, np, steps, a, b, c, workspace, workspace_bytes, sub_batch, flags, stream,
                  nullptr);
}

extern "C" int himuon_ns5_untile_apply_supported(int mp, int np, int tile_h, int tile_w, int steps, int flags,
                                                 int param_dtype) {
  const int family = flags & HIMUON_NS_FAMILY_MASK;
  return ns5_ba_supported(mp, np) && family == HIMUON_NS_FAMILY_AUTO && steps >= 2 && tile_h >= 1 &&
         tile_h <= tile_w && tile_w <= np && tile_h <= mp &&
         (param_dtype == HIMUON_DTYPE_F32 || param_dtype == HIMUON_DTYPE_BF16);
}

extern "C" int himuon_ns5_untile_apply(uint16_t* x, uint16_t* y, const float* inv, int64_t n_tiles, int mp, int np,
                                       int steps, float a, float b, float c, void* workspace,
                                       size_t workspace_bytes, int64_t sub_batch, int flags,
                                       const HimuonParamDesc* params_dev, int n_params, int64_t tile_begin,
                                       int tile_h, int tile_w, int param_dtype, const float* scale_alpha_dev,
                                       void* stream) {
  if (!himuon_ns5_untile_apply_supported(mp, np, tile_h, tile_w, steps, flags, param_dtype) || !params_dev ||
      n_params <= 0 || tile_begin < 0 || !scale_alpha_dev)
    return HIMUON_EINVAL;
  const BaUntile u{params_dev, n_params, tile_begin, tile_h, tile_w, param_dtype, scale_alpha_dev};
  return ns5_impl(x, y, inv, n_tiles, mp, np, steps, a, b, c, workspace, workspace_bytes, sub_batch, flags, stream,
                  &u);
}

// ---------------------------------------------------------------------------
// Allocation-free NS5: the A/B workspace is a file-scope device array (one
// copy per GPU, held until the process ends). Its device address is looked
// up once per device with that device current; host code uses only that
// address, never the array's name (a host-side stand-in).
// ---------------------------------------------------------------------------
namespace {
__device__ __align__(256) uint8_t scratch[HIMUON_NS_SCRATCH_BYTES];

constexpr int kMaxDevices = 64;
std::atomic<void*> g_scratch_dev[kMaxDevices];
std::mutex g_scratch_mu;

// Device address of this device's `scratch`, or nullptr (err set).
void* scratch_address(int* err) {
  int dev = 0;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) {
    *err = (int)e;
    return nullptr;
  }
  if (dev < 0 || dev >= kMaxDevices) {
    *err = HIMUON_EINVAL;
    return nullptr;
  }
  void* p = g_scratch_dev[dev].load(std::memory_order_acquire);
  if (p) return p;
  std::lock_guard<std::mutex> lock(g_scratch_mu);
  p = g_scratch_dev[dev].load(std::memory_order_relaxed);
  if (!p) {
    e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess || !p) {
      *err = e != hipSuccess ? (int)e : (int)hipErrorInvalidSymbol;
      return nullptr;
    }
    g_scratch_dev[dev].store(p, std::memory_order_release);
  }
  return p;
}
}  // namespace

extern "C" int himuon_lds_step(const HimuonParamDesc* params_dev, int n_params, int64_t tile_begin,
                               int64_t n_tiles, int tile_h, int tile_w, int dtype, int param_dtype, int steps,
                               float a, float b, float c, float eps, int flags, const float* scale_alpha_dev,
                               void* stream) {
  if (!params_dev || n_params <= 0 || tile_begin < 0 || n_tiles < 0 || steps < 0 || !scale_alpha_dev ||
      (flags & ~HIMUON_NS_ROUND_ONCE) || !lds_step_supported(tile_h, tile_w, dtype, param_dtype))
    return HIMUON_EINVAL;
  if (n_tiles == 0) return 0;
  lds_step_run(params_dev, n_params, tile_begin, n_tiles, tile_h, tile_w, dtype, param_dtype, steps, a, b, c,
               eps, (flags & HIMUON_NS_ROUND_ONCE) != 0, scale_alpha_dev, static_cast<hipStream_t>(stream));
  return (int)hipGetLastError();
}

extern "C" int himuon_reg_step(const HimuonParamDesc* params_dev, int n_params, int64_t tile_begin,
                               int64_t n_tiles, int tile_h, int tile_w, int dtype, int param_dtype, int steps,
                               float a, float b, float c, float eps, int flags, const float* scale_alpha_dev,
                               void* stream) {
  if (!params_dev || n_params <= 0 || tile_begin < 0 || n_tiles < 0 || steps < 0 || !scale_alpha_dev ||
      (flags & ~HIMUON_NS_ROUND_ONCE) || !reg_step_supported(tile_h, tile_w, dtype, param_dtype))
    return HIMUON_EINVAL;
  if (n_tiles == 0) return 0;
  reg_step_run(params_dev, n_params, tile_begin, n_tiles, tile_h, tile_w, dtype, param_dtype, steps, a, b, c,
               eps, (flags & HIMUON_NS_ROUND_ONCE) != 0, scale_alpha_dev, static_cast<hipStream_t>(stream));
  return (int)hipGetLastError();
}

extern "C" int himuon_ns_direct_supported(int M, int N, int dtype) {
  const bool rows = (M > 64 && N <= 128) || (M > 128 && N <= 256);
  return rows && M <= N && (dtype == HIMUON_DTYPE_F32 || dtype == HIMUON_DTYPE_BF16 || dtype == HIMUON_DTYPE_F16);
}

extern "C" int himuon_ns_direct(const void* g, void* out, int64_t batch, int M, int N, int dtype, int steps, float a,
                                float b, float c, float eps, int flags, void* stream) {
  if (!g || !out || batch < 0 || batch > 0x7fffffff || steps < 0 || (flags & ~HIMUON_NS_ROUND_ONCE) ||
      !himuon_ns_direct_supported(M, N, dtype))
    return HIMUON_EINVAL;
  if (batch == 0) return 0;
  const hipStream_t s = static_cast<hipStream_t>(stream);
  const bool ro = (flags & HIMUON_NS_ROUND_ONCE) != 0;
  if (N <= 128) ns_direct_lds_run(g, out, batch, M, N, dtype, steps, a, b, c, eps, ro, s);
  else ns_direct_reg_run(g, out, batch, M, N, dtype, steps, a, b, c, eps, ro, s);
  return (int)hipGetLastError();
}

extern "C" int himuon_ns5_noalloc(uint16_t* x, uint16_t* y, const float* inv, int64_t n_tiles, int mp,
                                  int np, int steps, float a, float b, float c, int flags, void* stream) {
  if (!x || !y || x == y || !inv || n_tiles < 0 || steps < 0 || mp <= 0 || np <= 0 || mp > np ||
      mp % HIMUON_NS_ALIGN || np % HIMUON_NS_ALIGN)
    return HIMUON_EINVAL;
  const size_t per_tile = himuon_ns5_workspace_bytes(1, mp, np);
  if (per_tile > HIMUON_NS_SCRATCH_BYTES) return HIMUON_ENOSPC;  // one tile's A and B do not fit
  if (n_tiles == 0) return 0;
  if (steps == 0)  // no workspace needed
    return himuon_ns5_ex(x, y, inv, n_tiles, mp, np, 0, a, b, c, nullptr, 0, n_tiles, flags, stream);
  int err = 0;
  void* ws = scratch_address(&err);
  if (!ws) return err;
  const int64_t sub_batch = (int64_t)(HIMUON_NS_SCRATCH_BYTES / per_tile);
  return himuon_ns5_ex(x, y, inv, n_tiles, mp, np, steps, a, b, c, ws, HIMUON_NS_SCRATCH_BYTES, sub_batch, flags,
                       stream);
}

extern "C" int himuon_ns5(uint16_t* x, uint16_t* y, const float* inv, int64_t n_tiles, int mp,
                          int np, int steps, float a, float b, float c, void* workspace,
                          size_t workspace_bytes, int64_t sub_batch, void* stream) {
  return himuon_ns5_ex(x, y, inv, n_tiles, mp, np, steps, a, b, c, workspace, workspace_bytes,
                       sub_batch, HIMUON_NS_FAMILY_AUTO, stream);
}

// ---------------------------------------------------------------------------
// One product on the faster block size. 256 x 256 blocks run one per CU, so r =
// blocks / CUs of them take ceil(r) rounds, full or not; 64 x 64 and 128 x 128
// blocks (ns_blk_product), two workgroups of 128 per CU, take a time that grows
// evenly with r: blk_rounds(), in those rounds. Beyond three rounds the 256 x 256
// blocks are ahead, or a few per cent behind, throughout. Below one round (r < 1)
// the 128 x 128 blocks win while they are one round themselves, two per CU, or
// little more.
//
// The constants are fitted to 1,689 products measured both ways (M 256 .. 8192,
// K up to 11 M, r 0.1 .. 8): the choice is within 0.6 % of always taking the faster
// one, 1.13 times as fast as 256 x 256 blocks alone, and more than 3 % behind those in
// four of the products. Points near the lines (us, smaller blocks / 256 x 256):
//
//   Apply M <= 256   269 of 256 x 256, r 1.05: 26 / 34      794, r 3.10: 75 / 68
//   Apply M <= 2048  42 of 1024 x 1024, r 2.62: 116 / 99    33, r 2.06: 90 / 96
//                    8 of 2048 x 2048, r 2.0: 153 / 124     5, r 1.25: 93 / 107
//   Apply beyond     5120 x 5120, r 1.56: 322 / 260         4096 x 4352, r 1.06: 184 / 198
//   Gram r < 1       13 of 1024 x 1024 (468 of 128): 25 / 36   17 (612): 35 / 33
//   Gram M < 512     269 of 256 x 256, r 1.05: 16 / 21      (or K < 1024)
//   Gram otherwise   33 of 1024 x 1024, r 1.29: 55 / 63     50, r 1.95: 76 / 70
//   Gram M >= 2560   7 of 3072 x 3072, r 2.13: 239 / 258    7 of 3072 x 12288: 1021 / 930
//   Gram M >= 5120   6144 x 6144, r 1.17: 289 / 306         7168 x 7168, r 1.59: 448 / 377
// ---------------------------------------------------------------------------
namespace {
double blk_rounds(int mode, int M, int K, double r) {
  if (mode == kApply) return M <= 256 ? 0.2 + 1.15 * r : M <= 2048 ? 0.2 + 1.25 * r : 0.05 + 1.56 * r;
  if (M >= 5120 || (M >= 2560 && K / 2 >= M)) return 1.55 * r;
  if (M >= 2560) return 1.33 * r;
  return (M >= 512 && K >= 1024 ? 1.26 : 1.3) * r;
}

bool smaller_blocks(int mode, const NsProduct& g) {
  if (g.M % 256 || g.N % 256 || g.K % 256) return true;
  const int64_t nb = g.M / 256, cus = num_cus();
  const int64_t items = g.ntiles * (mode == kApply ? nb * (g.N / 256) : nb * (nb + 1) / 2);
  if (items > 3 * cus) return false;
  if (items >= cus) return blk_rounds(mode, g.M, g.K, (double)items / cus) < (double)((items + cus - 1) / cus);
  // 128 x 128 blocks against one round of two per CU
  const int64_t blocks = mode == kApply ? 4 * items : g.ntiles * nb * (2 * nb + 1);
  const double rounds = blocks / (2.0 * cus);
  if (mode == kApply) return rounds <= (g.M <= 1024 ? 1.24 : 1.0);
  return rounds <= (g.M < 2560 ? 1.15 : 1.0);
}
}  // namespace

void ns_product(int mode, const NsProduct& g, hipStream_t s) {
  if (smaller_blocks(mode, g)) ns_blk_product(mode, g, s);
  else ns_stream_product(mode, g, s);
}

// ---------------------------------------------------------------------------
// The three NS products one at a time (the reference's kernel entry points
// XXT, ba_plus_cAA and fused_bmm_add): contiguous batches, dimensions
// multiples of 128; on the faster block size, or with the 128-block family on
// 64 x 64 or 128 x 128 blocks.
// ---------------------------------------------------------------------------
namespace {
bool stage_family(int flags, int* family) {
  *family = flags & HIMUON_NS_FAMILY_MASK;
  return !(flags & ~HIMUON_NS_FAMILY_MASK) &&
         (*family == HIMUON_NS_FAMILY_AUTO || *family == HIMUON_NS_FAMILY_BLOCK128);
}
}  // namespace

extern "C" int himuon_xxt(const uint16_t* x, uint16_t* out, int64_t batch, int M, int K, int flags,
                          void* stream) {
  int family = 0;
  if (!x || !out || batch < 0 || M <= 0 || K <= 0 || M % BM || K % BM || !stage_family(flags, &family))
    return HIMUON_EINVAL;
  if (batch == 0) return 0;
  const hipStream_t s = static_cast<hipStream_t>(stream);
  const int64_t xs = (int64_t)M * K, os = (int64_t)M * M;
  const NsProduct g{x, xs, K, x, xs, K, nullptr, 0, 0, out, os, M, M, M, K, batch, 1.f, 0.f, 0, nullptr};
  if (family == HIMUON_NS_FAMILY_AUTO) ns_product(kGramA, g, s);
  else ns_blk_product(kGramA, g, s);
  return (int)hipGetLastError();
}

extern "C" int himuon_ba_plus_caa(const uint16_t* a, uint16_t* out, int64_t batch, int M, float alpha,
                                  float beta, int flags, void* stream) {
  int family = 0;
  if (!a || !out || a == out || batch < 0 || M <= 0 || M % BM || !stage_family(flags, &family))
    return HIMUON_EINVAL;
  if (batch == 0) return 0;
  const hipStream_t s = static_cast<hipStream_t>(stream);
  const int64_t sq = (int64_t)M * M;
  const NsProduct g{a, sq, M, a, sq, M, a, sq, M, out, sq, M, M, M, M, batch, alpha, beta, 0, nullptr};
  if (family == HIMUON_NS_FAMILY_AUTO) ns_product(kGramB, g, s);
  else ns_blk_product(kGramB, g, s);
  return (int)hipGetLastError();
}

extern "C" int himuon_bmm_add(const uint16_t* b, const uint16_t* x, uint16_t* out, int64_t batch, int M, int N,
                              float a, int flags, void* stream) {
  int family = 0;
  const bool round_once = (flags & HIMUON_NS_ROUND_ONCE) != 0;
  if (!b || !x || !out || out == x || out == b || batch < 0 || M <= 0 || N <= 0 || M % BM || N % BM ||
      !stage_family(flags & ~HIMUON_NS_ROUND_ONCE, &family))
    return HIMUON_EINVAL;
  if (batch == 0) return 0;
  const hipStream_t s = static_cast<hipStream_t>(stream);
  const int64_t sq = (int64_t)M * M, rect = (int64_t)M * N;
  const NsProduct g{b, sq, M, x, rect, N, x, rect, N, out, rect, N, M, N, M, batch, 1.f, a, round_once ? 1 : 0, nullptr};
  if (family == HIMUON_NS_FAMILY_AUTO) ns_product(kApply, g, s);
  else ns_blk_product(kApply, g, s);
  return (int)hipGetLastError();
}

// ba_plus_cAA followed by fused_bmm_add as one kernel (ns5_ba.hip): B never
// leaves the CU. 512 x 512 only (the fused kernel's tile).
extern "C" int himuon_ba_bmm_add(const uint16_t* a, const uint16_t* x, uint16_t* out, int64_t batch, int M,
                                 int N, float alpha, float beta, float gamma, int flags, void* stream) {
  if (!a || !x || !out || out == x || out == a || batch < 0 || !ns5_ba_supported(M, N) ||
      (flags & ~HIMUON_NS_ROUND_ONCE))
    return HIMUON_EINVAL;
  if (batch == 0) return 0;
  if (!ns5_ba_run(a, x, out, nullptr, batch, gamma, beta, alpha, (flags & HIMUON_NS_ROUND_ONCE) != 0,
                  static_cast<hipStream_t>(stream)))
    return HIMUON_EINVAL;  // batch above kBaMaxTiles (32-bit work-item indices)
  return (int)hipGetLastError();
}
