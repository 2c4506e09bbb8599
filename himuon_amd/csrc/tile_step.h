// The memory passes of the kernels that hold an NS tile on chip for the whole
// optimizer step (lds_step_kernel in ns5_lds.hip, reg_step_kernel in
// ns5_reg.hip): momentum and gather of a plain N x N tile into LDS, and the
// untile with WD/LR from LDS. The per-element arithmetic is that of the
// separate gather and untile kernels (elem_ops.h).
//
// A thread's vectors (8 elements each) of the row-major N x N tile, in order:
// of the tile's 16384-element slabs it takes slab tid / 256 of every group of
// NT / 256 slabs, and in a slab the vectors tid % 256, + 256, .., + 1792. That
// is the gather kernel's order, so the sum of squares of a slab, summed per
// thread in this order and then over the slab's four waves, has its bits.
#pragma once

#include "elem_ops.h"
#include "lds_tiles.h"

template <int N, int NT>
struct StepGeo {
  static constexpr int VPR = N / 8;             // vectors per row
  static constexpr int VPT = N * VPR / NT;      // vectors per thread
  static constexpr int SLABS = VPT / 8;         // slabs per thread
  HM_DEV static int vec(int i, int tid) {       // tile vector of the thread's i-th
    return (i / 8) * (8 * NT) + (tid >> 8) * 2048 + (i % 8) * 256 + (tid & 255);
  }
};

struct TileAt {
  const HimuonParamDesc* P;
  int r, c;
};

HM_DEV TileAt tile_at(const HimuonParamDesc* __restrict__ params, int n_params, int64_t t) {
  const HimuonParamDesc* P = params + find_param(params, n_params, t);
  const int64_t lt = t - P->tile0;
  return TileAt{P, (int)(lt / P->C), (int)(lt % P->C)};
}

// Exactly one of UNT and GAT. UNT: untile with WD/LR of tile tu from X (X'
// of the NS iterations). GAT: momentum and gather of tile tg into X (bf16(e),
// not yet normalised); returns this thread's sum of squares of it. Both over
// the thread's slab s0 (0 .. SLABS - 1) of the tile; each thread reads and
// writes only its own vectors of X. BATCH: vectors whose loads are issued
// before any is used.
template <int N, int NT, int DT, int PDT, bool UNT, bool GAT, int BATCH>
HM_DEV float step_io(const HimuonParamDesc* __restrict__ params, int n_params, lds_u8* X, int64_t tu, int64_t tg,
                     int tile_h, int tile_w, const float* __restrict__ sa, int s0) {
#pragma clang fp contract(off)
  static_assert(UNT != GAT, "one tile pass per call");
  using Geo = StepGeo<N, NT>;
  constexpr int XCH = N / 8;
  static_assert(8 % BATCH == 0, "a batch stays inside a slab");
  TileAt U{nullptr, 0, 0}, G{nullptr, 0, 0};
  float s = 0.f, alpha = 0.f, sc = 0.f, mu = 0.f;
  bool has_mom = false, nesterov = false;
  if constexpr (UNT) {
    U = tile_at(params, n_params, tu);
    s = sa[2 * U.P->group];
    alpha = sa[2 * U.P->group + 1];
    sc = U.P->upd_scale;
  }
  if constexpr (GAT) {
    G = tile_at(params, n_params, tg);
    has_mom = G.P->momentum != nullptr;
    mu = G.P->mu;
    nesterov = G.P->nesterov != 0;
  }
  // (addresses from an opaque copy of the thread index: shared with the other
  // pass and kept live across the NS iterations they would not fit beside
  // those iterations' registers)
  const int tq = opaque_lane((int)threadIdx.x);
  float ssq = 0.f;
#pragma unroll 1
  for (int b0 = 8 * s0; b0 < 8 * s0 + 8; b0 += BATCH) {
    // phase 1: every global load of the batch (parameters of tile tu, or
    // grads and momentum of tile tg) before any is used
    float pv[BATCH][8], g[BATCH][8], m[BATCH][8];
    bool uok[BATCH], ufull[BATCH], fast[BATCH];
#pragma unroll
    for (int k = 0; k < BATCH; ++k) {
      const int v = Geo::vec(b0 + k, tq);
      const int i = v / Geo::VPR, j0 = (v % Geo::VPR) * 8;
      if constexpr (UNT) {
        const int64_t pr = (int64_t)U.r * tile_h + i, pc = (int64_t)U.c * tile_w + j0;
        const int64_t ou = pr * U.P->ld_upd + pc;
        uok[k] = i < tile_h && j0 < tile_w && pr < U.P->h && pc < U.P->w;
        ufull[k] = uok[k] && j0 + 8 <= tile_w && pc + 8 <= U.P->w;
        if (ufull[k]) load8<PDT>(U.P->update, ou, pv[k]);
      }
      if constexpr (GAT) {
        const int64_t pr = (int64_t)G.r * tile_h + i, pc = (int64_t)G.c * tile_w + j0;
        const int64_t og = pr * G.P->ld_grad + pc, om = pr * G.P->ld_mom + pc;
        fast[k] = i < tile_h && pr < G.P->h && j0 + 8 <= tile_w && pc + 8 <= G.P->w;
        if (fast[k]) {
          load8<DT>(G.P->grad, og, g[k]);
          if (has_mom) load8<DT>(G.P->momentum, om, m[k]);
        }
      }
    }
    // phase 2: the untile reads X' of vector v, or the gather writes it
#pragma unroll
    for (int k = 0; k < BATCH; ++k) {
      const int v = Geo::vec(b0 + k, tq);
      const int i = v / Geo::VPR, j0 = (v % Geo::VPR) * 8;
      lds_u32x4* const px = reinterpret_cast<lds_u32x4*>(X + lds_pos(i, v % Geo::VPR, XCH));
      if constexpr (UNT) {
        if (uok[k]) {
          const u32x4_t w = *px;
          float y[8];
#pragma unroll
          for (int e2 = 0; e2 < 4; ++e2) {
            y[2 * e2] = sc * bf16_to_f32(w[e2] & 0xffffu);
            y[2 * e2 + 1] = sc * __uint_as_float(w[e2] & 0xffff0000u);
          }
          const int64_t pr = (int64_t)U.r * tile_h + i, pc = (int64_t)U.c * tile_w + j0;
          const int64_t ou = pr * U.P->ld_upd + pc;
          if (ufull[k]) {  // put8<true>'s full form, its load issued above
#pragma unroll
            for (int e = 0; e < 8; ++e)
              pv[k][e] = __builtin_fmaf(alpha, round_to<PDT>(y[e]), round_to<PDT>(pv[k][e] * s));
            store8<PDT>(U.P->update, ou, pv[k]);
          } else {
            const int valid = (int)min<int64_t>(min(8, tile_w - j0), U.P->w - pc);
            put8<true, PDT>(*U.P, ou, y, false, valid, sa);
          }
        }
      }
      if constexpr (GAT) {
        const int64_t pr = (int64_t)G.r * tile_h + i, pc = (int64_t)G.c * tile_w + j0;
        const int64_t og = pr * G.P->ld_grad + pc, om = pr * G.P->ld_mom + pc;
        float x[8];
        if (fast[k]) {
#pragma unroll
          for (int e = 0; e < 8; ++e) x[e] = momentum_elem<DT>(g[k][e], &m[k][e], mu, nesterov, has_mom);
          if (has_mom) store8<DT>(G.P->momentum, om, m[k]);
        } else {
          const bool row_ok = i < tile_h && pr < G.P->h;
#pragma unroll
          for (int e = 0; e < 8; ++e) {
            x[e] = 0.f;
            if (row_ok && j0 + e < tile_w && pc + e < G.P->w) {
              const float gv = load_elem<DT>(G.P->grad, og + e);
              float mv = has_mom ? load_elem<DT>(G.P->momentum, om + e) : 0.f;
              x[e] = momentum_elem<DT>(gv, &mv, mu, nesterov, has_mom);
              if (has_mom) store_elem<DT>(G.P->momentum, om + e, mv);
            }
          }
        }
        uint32_t h[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          h[e] = f32_to_bf16(x[e]);
          const float f = bf16_to_f32(h[e]);
          ssq = fmaf(f, f, ssq);
        }
        *px = u32x4_t{pack2(h[0], h[1]), pack2(h[2], h[3]), pack2(h[4], h[5]), pack2(h[6], h[7])};
      }
    }
  }
  return ssq;
}

// newton_schulz on a contiguous batch of rows x cols matrices (rows <= cols <=
// N), matrix t: slab s0 of it as bf16 into X, zero padded to N x N; returns
// this thread's sum of squares of it.
template <int N, int NT, int DT, int BATCH>
HM_DEV float direct_load(const void* __restrict__ g, lds_u8* X, int64_t t, int rows, int cols, int s0) {
#pragma clang fp contract(off)
  using Geo = StepGeo<N, NT>;
  static_assert(8 % BATCH == 0, "a batch stays inside a slab");
  const int tq = opaque_lane((int)threadIdx.x);
  const int64_t base = t * (int64_t)rows * cols;
  float ssq = 0.f;
#pragma unroll 1
  for (int b0 = 8 * s0; b0 < 8 * s0 + 8; b0 += BATCH) {
    float x[BATCH][8];
    bool full[BATCH];
#pragma unroll
    for (int k = 0; k < BATCH; ++k) {
      const int v = Geo::vec(b0 + k, tq), i = v / Geo::VPR, j0 = (v % Geo::VPR) * 8;
      full[k] = i < rows && j0 + 8 <= cols;
      if (full[k]) load8<DT>(g, base + (int64_t)i * cols + j0, x[k]);
    }
#pragma unroll
    for (int k = 0; k < BATCH; ++k) {
      const int v = Geo::vec(b0 + k, tq), i = v / Geo::VPR, j0 = (v % Geo::VPR) * 8;
      if (!full[k]) {
#pragma unroll
        for (int e = 0; e < 8; ++e)
          x[k][e] = i < rows && j0 + e < cols ? load_elem<DT>(g, base + (int64_t)i * cols + j0 + e) : 0.f;
      }
      uint32_t h[8];
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        h[e] = f32_to_bf16(x[k][e]);
        const float f = bf16_to_f32(h[e]);
        ssq = fmaf(f, f, ssq);
      }
      *reinterpret_cast<lds_u32x4*>(X + lds_pos(i, v % Geo::VPR, N / 8)) =
          u32x4_t{pack2(h[0], h[1]), pack2(h[2], h[3]), pack2(h[4], h[5]), pack2(h[6], h[7])};
    }
  }
  return ssq;
}

// Slab s0 of X to matrix t of the contiguous output batch.
template <int N, int NT, int DT>
HM_DEV void direct_store(void* __restrict__ out, const lds_u8* X, int64_t t, int rows, int cols, int s0) {
  using Geo = StepGeo<N, NT>;
  const int tq = opaque_lane((int)threadIdx.x);
  const int64_t base = t * (int64_t)rows * cols;
#pragma unroll
  for (int k = 8 * s0; k < 8 * s0 + 8; ++k) {
    const int v = Geo::vec(k, tq), i = v / Geo::VPR, j0 = (v % Geo::VPR) * 8;
    if (i >= rows || j0 >= cols) continue;
    const u32x4_t w = *reinterpret_cast<lds_cu32x4*>(X + lds_pos(i, v % Geo::VPR, N / 8));
    float y[8];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      y[2 * e] = bf16_to_f32(w[e] & 0xffffu);
      y[2 * e + 1] = __uint_as_float(w[e] & 0xffff0000u);
    }
    const int64_t o = base + (int64_t)i * cols + j0;
    if (j0 + 8 <= cols) {
      store8<DT>(out, o, y);
    } else {
#pragma unroll
      for (int e = 0; e < 8; ++e)
        if (j0 + e < cols) store_elem<DT>(out, o + e, y[e]);
    }
  }
}
