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
// X stays in registers and the Gram products' 36 lower tiles are split 5, 5, 5, 5,
// 4, 4, 4, 4 over the waves (9 per SIMD, wave w sharing SIMD w % 4 with wave w +
// 4), each wave working from four row fragments per k-step (ns_reg.h).
#include "ns_reg.h"
#include "tile_step.h"

namespace {

constexpr int T = 256;          // tile edge
constexpr int NT = 512;         // threads: eight waves
constexpr int CH = T / 8;       // 16-byte chunks per row
constexpr int LDS_BYTES = T * T * 2;
// 8-element vectors whose loads are in flight per thread in the step's memory
// passes (grad and momentum: 16 VGPRs each, parameters: 8 or 4)
constexpr int GAT_BATCH = 4, UNT_BATCH = 8;

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
  ns_reg::reg_iterations<T>(L, sc, steps, ca, cb, cc, round_once);
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
// 4 in the untile's: within 0.6 %. (256 VGPRs and one spilled, here and in
// ns_direct_reg_kernel; ns5_reg_kernel takes 203.)
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
  ns_reg::reg_iterations<T>(L, s_inv, steps, ca, cb, cc, round_once);
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
  ns_reg::reg_iterations<T>(L, s_inv, steps, ca, cb, cc, round_once);
#pragma unroll 1
  for (int s = 0; s < 2; ++s) direct_store<T, NT, DT>(out, L, t, rows, cols, s);
}

}  // namespace

void ns_direct_reg_run(const void* g, void* out, int64_t cnt, int rows, int cols, int dtype, int steps, float a,
                       float b, float c, float eps, bool round_once, hipStream_t s) {
  const int64_t bytes = (int64_t)rows * cols * (dtype == HIMUON_DTYPE_F32 ? 4 : 2);
  const auto run = [&](auto kernel) {
    per_launch(cnt, NT, [&](int64_t off, int64_t n) {
      hipLaunchKernelGGL(kernel, dim3((unsigned)n), dim3(NT), 0, s, static_cast<const char*>(g) + off * bytes,
                         static_cast<char*>(out) + off * bytes, n, rows, cols, steps, a, b, c, eps, round_once ? 1 : 0);
    });
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
  per_launch(cnt, NT, [&](int64_t off, int64_t n) {
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
  });
}

bool ns5_reg_supported(int mp, int np) { return mp == T && np == T; }

void ns5_reg_run(uint16_t* x, uint16_t* y, const float* inv, int64_t cnt, int steps, float a, float b, float c,
                 bool round_once, hipStream_t s) {
  uint16_t* out = (steps & 1) ? y : x;
  per_launch(cnt, NT, [&](int64_t off, int64_t n) {
    hipLaunchKernelGGL(ns5_reg_kernel, dim3((unsigned)n), dim3(NT), 0, s, x + off * T * T, out + off * T * T,
                       inv + off, n, steps, a, b, c, round_once ? 1 : 0);
  });
}
