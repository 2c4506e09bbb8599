// The three NS5 products on 128 x 128 (BT = 128) or 64 x 64 output blocks, for NS
// tiles whose padded edges are any multiples of 128:
//
//   GramA : C = A = bf16(X X^T)            P = Q = X (rows, K = n)   lower blocks + mirror
//   GramB : C = B = bf16(c A A^T + b A)    P = Q = A (rows, K = m)   lower blocks + mirror
//   Apply : C = X' = bf16(bf16(B X) + a X) P = B (rows, K = m), Q = X read as [k][j]
// (ns5_smem.py:89-101, XXT.py:55-75, ba_plus_cAA.py:58-85, fused_bmm_add.py:65-88).
//
// One workgroup per block: 4 waves in 2 x 2, each 64 x 64 as 2 x 2 (BT = 64: 32 x
// 32 as one) v_mfma_f32_32x32x16_bf16 tiles; two workgroups fit a CU at BT = 128
// (64 KiB of LDS each), five at BT = 64 (32 KiB), so one's MFMAs run while another
// waits at a barrier, starts or stores. K advances in units of 64, straight from global memory into one of
// two LDS slots (32 KiB each at BT = 128), one unit ahead of the MFMAs; the epilogue operand R
// (A for GramB, X for Apply) follows as one more unit. The swapped MFMA
// operand order and the mirrored store are those of the 256-block kernels
// (ns5_stream.hip), and every element sums its k terms in one accumulator in
// ascending order as there.
//
// What bounds it: the operand stream from L2 (32 KiB per 64 MFMAs; without
// the loads a large batch runs 1.2 to 1.6 times as fast, without the MFMAs or
// the fragment reads 1.06 to 1.4 times). So a unit is 64 wide: its rows are
// whole 128-byte lines, which units of 32 fetched twice (1024 x 1024 GramA of
// 56 matrices 82 against 91 us, Apply 164 against 181 us, with five such
// slots), and two slots at two workgroups per CU are worth more than three
// slots at one (101 and 193 us). Against the register-staged kernels this
// replaced, GramA / GramB / Apply of 12 matrices of 896 x 2432: 42 / 21 / 64
// against 58 / 46 / 150 us; 512 of 384 x 384: 73 / 80 / 122 against 154 / 230
// / 221 us.
#include "lds_tiles.h"

namespace {

constexpr int NT = 256;           // four waves
constexpr int BK = 64;            // K per unit

// Chunk swizzles (16-byte chunk index XOR a function of the row): rows of 128
// bytes (panels of P / Q; R and the output staging of some block edges): 16
// consecutive rows of one chunk on distinct bank groups; likewise rows of 64
// and 256 bytes; X panel rows of 256 or 128 bytes: the 4 rows x 4 chunks of a
// transposing read.
template <int BYTES>
HM_DEV int swz(int r) {
  return BYTES == 256 ? r & 15 : BYTES == 128 ? (r >> 1) & 7 : (r >> 2) & 3;
}
template <int BYTES>
HM_DEV int swz_x(int r) {
  return BYTES == 256 ? 4 * (r & 3) : 4 * ((r >> 1) & 1);
}

// One block. DIAG: Gram diagonal block, Q = P (one panel streamed), no mirror.
// SC: the X operand is the raw tile, every X value replaced by bf16(x inv) as
// it enters the computation.
template <int MODE, bool SC, bool DIAG, int BT>
HM_DEV void blk_item(const NsProduct& g, lds_u8* lds, int64_t tile, int bi, int bj) {
  constexpr bool kTr = MODE == kApply;
  constexpr int HALF = BT * BK * 2, SLOT = 2 * HALF;  // bytes of an operand's unit, of a unit
  constexpr int XB = BT * 2;                          // bytes per row of the X panel and of R
  constexpr int XR = 1024 / XB, XC = XB / 16;         // their rows per 1 KiB, chunks per row
  constexpr int PI = BT / 32;                         // panel loads per wave
  constexpr int WT = BT / 64, WC = BT / 2;            // MFMA tiles, rows / columns per wave
  constexpr bool kR = MODE != kGramA;  // an epilogue operand
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave >> 1, wn = wave & 1;
  const int l32 = lane & 31, hi = lane >> 5;
  const int nk = g.K / BK, units = nk + kR;
  float xs = 1.f;
  if constexpr (SC) xs = uniform_load_f32(g.inv, tile);

  // ---- loaders: wave instruction n = 4 i + wave fills 1 KiB n of a panel ----------
  // Row panel: rows 8 n .. + 7; lane l lands at row 8 n + l / 8, position
  // l % 8. X panel: XR k-rows, lane l at row XR n + l / XC, position l % XC.
  const int prl = 8 * wave + (lane >> 3), pch = (lane & 7) ^ swz<128>(prl);
  const uint16_t* const psrc = g.P + tile * g.p_bs + (int64_t)(bi * BT + prl) * g.ldp + pch * 8;
  const uint16_t* qsrc;
  int64_t qstep, qunit;
  if constexpr (kTr) {
    const int xr = XR * wave + lane / XC;
    qsrc = g.Q + tile * g.q_bs + (int64_t)xr * g.ldq + bj * BT + ((lane & (XC - 1)) ^ swz_x<XB>(xr)) * 8;
    qstep = 4 * XR * (int64_t)g.ldq;
    qunit = BK * (int64_t)g.ldq;
  } else {
    qsrc = g.Q + tile * g.q_bs + (int64_t)(bj * BT + prl) * g.ldq + pch * 8;
    qstep = 32 * (int64_t)g.ldq;
    qunit = BK;
  }
  const int64_t pstep = 32 * (int64_t)g.ldp;
  const uint32_t wdst = (uint32_t)(uintptr_t)lds + wave * 1024;
  auto issue = [&](int v, int slot) {
    const uint32_t d = wdst + slot * SLOT;
    if (v < nk) {
#pragma unroll
      for (int i = 0; i < PI; ++i) dma16(psrc + i * pstep + v * BK, d + i * 4096);
      if constexpr (!DIAG) {
#pragma unroll
        for (int i = 0; i < PI; ++i) dma16(qsrc + i * qstep + v * qunit, d + HALF + i * 4096);
      }
    } else if constexpr (kR) {  // R: the block's rows
      const uint16_t* const r0 = g.R + tile * g.r_bs + (int64_t)(bi * BT) * g.ldr + bj * BT;
#pragma unroll
      for (int i = 0; i < BT / XR / 4; ++i) {
        const int r = XR * (4 * i + wave) + lane / XC;
        dma16(r0 + (int64_t)r * g.ldr + ((lane & (XC - 1)) ^ swz<XB>(r)) * 8, d + i * 4096);
      }
    }
  };
  // GramA of the first iteration: the wave's own pieces of a unit scaled in
  // LDS, after its wait for them and before the barrier that publishes them
  auto scale_unit = [&](int slot) {
    if constexpr (SC && MODE == kGramA) {
      asm volatile("" ::: "memory");  // the reads below follow the vmcnt wait
      lds_u8* const d = lds + slot * SLOT + wave * 1024 + 16 * lane;
#pragma unroll
      for (int i = 0; i < (DIAG ? PI : 2 * PI); ++i) {
        lds_u32x4* const p = reinterpret_cast<lds_u32x4*>(d + i * 4096);
        *p = scale8_rne(*p, xs);
      }
    }
  };

  // ---- fragments: fb rows i of P, fa rows (columns) j of Q --------------------------
  const int sp = swz<128>(l32);
  const int prow = (wm * WC + l32) * 128, qrow = (wn * WC + l32) * 128;
  const int tr_krow = tr_krow_of(lane), tr_col = tr_col_of(lane);
  const uint32_t tr_lane = HALF + tr_krow * XB + (tr_col & 7) * 2;
  auto frags = [&](int slot, int ks, u32x4_t(&fa)[WT], u32x4_t(&fb)[WT]) {
    const lds_u8* s = lds + slot * SLOT;
    const int pos = ((2 * ks + hi) ^ sp) * 16;
#pragma unroll
    for (int t = 0; t < WT; ++t) fb[t] = *reinterpret_cast<lds_cu32x4*>(s + prow + t * 4096 + pos);
#pragma unroll
    for (int t = 0; t < WT; ++t) {
      if constexpr (kTr) {  // (rows kr and kr + 4 have one swizzle)
        const int ch = (wn * (WC / 8) + 4 * t + (tr_col >> 3)) ^ swz_x<XB>(tr_krow);
        const uint32_t off = tr_lane + 16 * ks * XB + ch * 16;
        const u32x2_t l2 = read_tr(s, off), u2 = read_tr(s, off + 4 * XB);
        fa[t] = u32x4_t{l2[0], l2[1], u2[0], u2[1]};
        if constexpr (SC) fa[t] = scale8_rne(fa[t], xs);
      } else {
        fa[t] = *reinterpret_cast<lds_cu32x4*>((DIAG ? s : s + HALF) + qrow + t * 4096 + pos);
      }
    }
  };
  f32x16_t acc[WT][WT];
#pragma unroll
  for (int a = 0; a < WT; ++a)
#pragma unroll
    for (int b = 0; b < WT; ++b)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[a][b][e] = 0.f;
  auto mma = [&](const u32x4_t(&fa)[WT], const u32x4_t(&fb)[WT]) {
#pragma unroll
    for (int tj = 0; tj < WT; ++tj)
#pragma unroll
      for (int ti = 0; ti < WT; ++ti) acc[tj][ti] = mfma(fa[tj], fb[ti], acc[tj][ti]);
  };

  // ---- K loop ----------------------------------------------------------------------
  // Unit u is in slot u % 2. Each k-step's fragments are read ahead of the
  // MFMAs of the step before it, across units too: before its last MFMAs of
  // unit u a wave waits for its own loads of unit u + 1, and the barrier
  // publishes that unit and frees the other slot (every wave's fragments of
  // unit u have landed), which receives unit u + 2.
  issue(0, 0);
  wait_vm<0>();
  scale_unit(0);
  lds_barrier();
  issue(1, 1);  // (nk >= 2)
  u32x4_t fa0[WT], fb0[WT], fa1[WT], fb1[WT];
  frags(0, 0, fa0, fb0);
#pragma unroll 1
  for (int u = 0; u < nk; ++u) {
    const int slot = u & 1;
    frags(slot, 1, fa1, fb1);
    __builtin_amdgcn_sched_barrier(0);
    mma(fa0, fb0);
    __builtin_amdgcn_sched_barrier(0);
    frags(slot, 2, fa0, fb0);
    __builtin_amdgcn_sched_barrier(0);
    mma(fa1, fb1);
    __builtin_amdgcn_sched_barrier(0);
    frags(slot, 3, fa1, fb1);
    __builtin_amdgcn_sched_barrier(0);
    mma(fa0, fb0);
    __builtin_amdgcn_sched_barrier(0);
    if (u + 1 < nk) {
      wait_vm<0>();
      scale_unit(slot ^ 1);
      lds_barrier();
      if (u + 2 < units) issue(u + 2, slot);
      frags(slot ^ 1, 0, fa0, fb0);
      __builtin_amdgcn_sched_barrier(0);
    }
    mma(fa1, fb1);
    __builtin_amdgcn_sched_barrier(0);
  }

  // ---- epilogue --------------------------------------------------------------------
  // out[ti][tj][q]: 4 bf16 of C[i][j .. j + 3], i = wm WC + 32 ti + l32,
  // j = wn WC + 32 tj + 8 q + 4 hi (block-local).
  u32x2_t out[WT][WT][4];
  wait_vm<0>();
  lds_barrier();  // R is in; every fragment read is done
#pragma unroll
  for (int ti = 0; ti < WT; ++ti)
#pragma unroll
    for (int tj = 0; tj < WT; ++tj)
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        float y[4];
        if constexpr (kR) {
          const int il = wm * WC + 32 * ti + l32, ch = wn * (WC / 8) + 4 * tj + q;
          const u32x2_t rv = *reinterpret_cast<lds_cu32x2*>(lds + (nk & 1) * SLOT + il * XB +
                                                            ((ch ^ swz<XB>(il)) * 16) + hi * 8);
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            float x = bf16_to_f32(half16(rv[e >> 1], e & 1));
            if constexpr (SC) x = bf16_to_f32(pk_bf16(x * xs, 0.f) & 0xffffu);
            const float v = acc[tj][ti][4 * q + e];
            if constexpr (MODE == kApply)
              y[e] = fmaf(g.beta, x, g.round_once ? v : bf16_to_f32(pk_bf16(v, 0.f) & 0xffffu));
            else
              y[e] = fmaf(g.beta, x, g.alpha * v);
          }
        } else {
#pragma unroll
          for (int e = 0; e < 4; ++e) y[e] = acc[tj][ti][4 * q + e];
        }
        out[ti][tj][q] = u32x2_t{pk_bf16(y[0], y[1]), pk_bf16(y[2], y[3])};
      }
  if constexpr (kR) lds_barrier();  // every R read is done
  // Staging: each wave's WC x WC result in its own LDS (LDS operations of a
  // wave execute in order), then whole rows, 16 bytes per lane.
  constexpr int SB = WC * 2, SC16 = SB / 16, SR = 64 / SC16;  // row bytes, chunks, rows per store
  lds_u8* const W = lds + wave * (WC * SB);
  const int srow = lane / SC16, sch = lane % SC16;
  uint16_t* const Ct = g.C + tile * g.c_bs;
  auto store_rows = [&](uint16_t* dst) {
#pragma unroll
    for (int n = 0; n < WC / SR; ++n) {
      const int r = SR * n + srow;
      const u32x4_t v = *reinterpret_cast<lds_cu32x4*>(W + r * SB + ((sch ^ swz<SB>(r)) * 16));
      *reinterpret_cast<u32x4_t*>(dst + (int64_t)r * g.ldc + sch * 8) = v;
    }
  };
#pragma unroll
  for (int ti = 0; ti < WT; ++ti)
#pragma unroll
    for (int tj = 0; tj < WT; ++tj)
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int r = 32 * ti + l32, ch = 4 * tj + q;
        *reinterpret_cast<lds_u32x2*>(W + r * SB + ((ch ^ swz<SB>(r)) * 16) + hi * 8) = out[ti][tj][q];
      }
  store_rows(Ct + (int64_t)(bi * BT + wm * WC) * g.ldc + bj * BT + wn * WC);
  if constexpr (MODE != kApply && !DIAG) {
    // mirror: after the quad transpose lane (a = l32 / 4, k = l32 % 4) holds
    // C^T[j][i .. i + 3], j = 32 tj + 8 q + 4 hi + k, i = 32 ti + 4 a
    const int k = lane & 3, a = l32 >> 2;
#pragma unroll
    for (int ti = 0; ti < WT; ++ti)
#pragma unroll
      for (int tj = 0; tj < WT; ++tj)
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const int r = 32 * tj + 8 * q + 4 * hi + k, ch = 4 * ti + (a >> 1);
          *reinterpret_cast<lds_u32x2*>(W + r * SB + ((ch ^ swz<SB>(r)) * 16) + (a & 1) * 8) =
              quad_transpose(out[ti][tj][q], k);
        }
    store_rows(Ct + (int64_t)(bj * BT + wn * WC) * g.ldc + bi * BT + wm * WC);
  }
}

template <int MODE, bool SC, int BT>
__global__ __launch_bounds__(NT, 2) void ns_blk_kernel(NsProduct g) {
  __shared__ __attribute__((aligned(1024))) uint8_t lds[8 * BT * BK];
  const int nbi = g.M / BT, nbj = g.N / BT;
  const int per_tile = MODE == kApply ? nbi * nbj : nbi * (nbi + 1) / 2;
  const int64_t total = g.ntiles * per_tile;
  const int64_t item = xcd_item(total);
  if (item >= total) return;
  const int64_t tile = item / per_tile;
  const int p = (int)(item - tile * per_tile);
  if constexpr (MODE == kApply) {
    blk_item<MODE, SC, false, BT>(g, (lds_u8*)lds, tile, p / nbj, p % nbj);
  } else {
    int bi = 0;
    while ((bi + 1) * (bi + 2) / 2 <= p) ++bi;
    const int bj = p - bi * (bi + 1) / 2;
    if (bi == bj) blk_item<MODE, SC, true, BT>(g, (lds_u8*)lds, tile, bi, bj);
    else blk_item<MODE, SC, false, BT>(g, (lds_u8*)lds, tile, bi, bj);
  }
}

template <int BT>
void launch(int mode, const NsProduct& g, hipStream_t s) {
  const int64_t nbi = g.M / BT, nbj = g.N / BT;
  const int64_t items = g.ntiles * (mode == kApply ? nbi * nbj : nbi * (nbi + 1) / 2);
  const dim3 grid((unsigned)xcd_grid(items)), block(NT);
  const bool sc = g.inv != nullptr;
  if (mode == kGramA) {
    if (sc) hipLaunchKernelGGL((ns_blk_kernel<kGramA, true, BT>), grid, block, 0, s, g);
    else hipLaunchKernelGGL((ns_blk_kernel<kGramA, false, BT>), grid, block, 0, s, g);
  } else if (mode == kGramB) {
    hipLaunchKernelGGL((ns_blk_kernel<kGramB, false, BT>), grid, block, 0, s, g);
  } else {
    if (sc) hipLaunchKernelGGL((ns_blk_kernel<kApply, true, BT>), grid, block, 0, s, g);
    else hipLaunchKernelGGL((ns_blk_kernel<kApply, false, BT>), grid, block, 0, s, g);
  }
}

}  // namespace

// 64 x 64 blocks where 128 x 128 ones would leave much of the chip idle: a
// workgroup alone on its CU is bound by its own operand stream (about 55 GB/s
// of it), which a smaller block shortens. One 1024 x 1024 matrix 7.7 / 7.9 /
// 8.1 against 12.4 / 13.5 / 12.7 us for the three products (36 and 64 blocks of
// 128), GramA of one 1024 x 3072 24 against 34 us, of 4 1024 x 1024 (144 blocks)
// 12.3 against 13.5; Apply of those (256 blocks) 15.6 against 14.8, all three of
// one 2560 x 2560 (210 and 400) 40 / 39 / 68 against 30 / 31 / 44. Gram products
// of 256 rows with K = 256 stay short enough for 64 x 64 (10 of 16 blocks
// computed instead of 3 of 4): 512 of them 29.5 against 34.7 us.
void ns_blk_product(int mode, const NsProduct& g, hipStream_t s) {
  if (!dma_aligned(g.P, g.Q, g.R)) return ns_any_product(mode, g, s);
  const int64_t nbi = g.M / 128, nbj = g.N / 128;
  const int64_t items = g.ntiles * (mode == kApply ? nbi * nbj : nbi * (nbi + 1) / 2);
  const bool short_gram = mode != kApply && g.K <= 256 && items < (1 << 21);  // a grid holds 2^24 workgroups
  if (items <= num_cus() * 5 / 8 || short_gram) launch<64>(mode, g, s);
  else launch<128>(mode, g, s);
}
