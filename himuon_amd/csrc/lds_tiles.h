// LDS layouts and MFMA fragment reads shared by the kernels that keep an NS
// tile on chip through its iterations (ns5_lds.hip, ns5_reg.hip).
#pragma once

#include "ns5_kernels.h"

typedef short v4i16 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) v4i16 lds_v4i16;
typedef __attribute__((address_space(3))) u32x4_t lds_u32x4;

HM_DEV uint32_t lds_pos(int r, int ch, int chunks) {
  const int sw = ((r & 3) << 2) | ((r >> 2) & 3);
  return (uint32_t)(r * chunks + (ch ^ sw)) * 16u;
}

// Stored lower 32x32 tile (ti >= tj) of a symmetric matrix of 32-row tiles:
// byte offset of 16-byte chunk ch (columns 8 ch ..) of its row r.
constexpr int TRI_TILE = 32 * 32 * 2;
constexpr int tri_bytes(int row_tiles) { return row_tiles * (row_tiles + 1) / 2 * TRI_TILE; }
HM_DEV uint32_t tri_pos(int ti, int tj, int r, int ch) {
  return (uint32_t)((ti * (ti + 1) / 2 + tj) * TRI_TILE + r * 64 + ((ch ^ ((r >> 2) & 3)) << 4));
}

// Transposing read: 4 bf16 of the 8-byte row segment at `off`, redistributed
// across each group of 16 lanes (lane 4a + b receives element b of the
// segments addressed by lanes a, a + 4, a + 8, a + 12).
HM_DEV u32x2_t read_tr(const lds_u8* base, uint32_t off) {
  const v4i16 r = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4i16*)(base + off));
  return __builtin_bit_cast(u32x2_t, r);
}

// The lane index, opaque to the optimiser: addresses derived from it are
// formed inside each phase instead of being hoisted out of the iteration loop
// for all four per-wave variants at once (which would not fit the registers).
HM_DEV int opaque_lane(int v) {
  asm volatile("" : "+v"(v));
  return v;
}

// Row fragment of a symmetric matrix S stored as its lower tiles: lane (l32,
// hi) receives S[32 R + l32][16 ks + 8 hi .. + 7] (the MFMA operand of row
// tile R, k-step ks). Column tile k = ks / 2 > R is read from the stored tile
// (k, R) as the transposing reads of the X operand do.
template <int R, int KS>
HM_DEV u32x4_t tri_frag(const lds_u8* S, int l32, int hi, int tr_krow, int tr_col) {
  constexpr int TK = KS >> 1;
  if constexpr (TK <= R) {
    return *reinterpret_cast<lds_cu32x4*>(S + tri_pos(R, TK, l32, 2 * (KS & 1) + hi));
  } else {
    const int kr = 16 * (KS & 1) + tr_krow;
    const u32x2_t l2 = read_tr(S, tri_pos(TK, R, kr, tr_col >> 3) + (tr_col & 7) * 2);
    const u32x2_t u2 = read_tr(S, tri_pos(TK, R, kr + 4, tr_col >> 3) + (tr_col & 7) * 2);
    return u32x4_t{l2[0], l2[1], u2[0], u2[1]};
  }
}

// Transposing-read lane roles (the X operand of Apply, the upper fragments of
// A and B): lane (a', b') of each 16-lane group addresses k-row 8 hi + a' (+ 4
// for the second read) and columns 16 ((lane >> 4) & 1) + 4 b' .. + 3 of a
// 32-column tile.
HM_DEV int tr_krow_of(int lane) { return 8 * (lane >> 5) + ((lane & 15) >> 2); }
HM_DEV int tr_col_of(int lane) { return 16 * ((lane >> 4) & 1) + 4 * (lane & 3); }
