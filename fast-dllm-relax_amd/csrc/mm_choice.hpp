// Which blocks a large-M projection runs on, and in how many k splits: host code without any GPU header, compiled
// into gemm.hip's launch planning and checked on the CPU (tests/mm_choice_check.cpp).
#pragma once
#include <algorithm>

namespace fdllm {

// The projections; their launch configurations are in gemm.hip.
enum GemmCfg : int { CFG_QKV = 0, CFG_OPROJ = 1, CFG_GATE_UP = 2, CFG_DOWN = 3, CFG_LM_HEAD = 4 };

// How large-M launches are planned.  target_wgs / min_stages: k is split only while the launch has fewer
// than target_wgs workgroups, and only into splits of at least min_stages stages.  wr_ops: the
// projections (bit cfg) that may take the register-weight kernel's large blocks, from wr_min_rows rows (0: the
// row counts where they measured faster than the LDS-staged and streaming kernels, mm_choice).
struct MmPolicy {
  int cus = 256;  // compute units
  int target_wgs = 256;
  int min_stages = 8;
  int wr_ops = (1 << CFG_QKV) | (1 << CFG_OPROJ) | (1 << CFG_GATE_UP) | (1 << CFG_DOWN) | (1 << CFG_LM_HEAD);
  int wr_min_rows = 0;
  int wr_small_ops = (1 << CFG_QKV) | (1 << CFG_OPROJ);  // take the 64 x 128 register-weight blocks below the 128 x 256 ones
  // gate_up / down below 1024 rows: -1 the measured choice, else bit 0 / 1 the 64 x 128 register-weight blocks,
  // bit 2 / 3 the 128 x 128 ones (0: the LDS-staged kernels)
  int wr_ffn = -1;
  int force_split = 0;  // > 1: this k split whenever it divides the stages (the fused o_proj + norm)
  int wr3 = 1;          // o_proj / down at the register-weight thresholds: 128 x 192 blocks (0: 128 x 256)
  int wt8 = 1;  // LDS-staged 128 x 192 blocks of eight waves (bit 0 gate_up, bit 1 down) instead of four
  int wt256 = 512;  // gate_up from 257 up to this many rows on LDS-staged 256 x 192 blocks of eight waves
  // the streaming lm_head of up to 32 rows: the column groups past the last whole round over this many
  // compute units (one group per unit per round) split k up to 3 ways, so that every unit streams about
  // the same bytes (0: off)
  int lm_tail_cus = 0;
  // one-shot projections (bit cfg) of 17 to 32 rows run as two 16-row m-chunks: each workgroup takes in
  // half the activations for the same weight tile
  int os_half = (1 << CFG_QKV) | (1 << CFG_OPROJ);
};

// The large-M kernels: LDS-staged gemm_mm_kernel (SMALL, WIDE, WIDE_D with weights two stages ahead, BIG) and
// gemm_wt_kernel (WT of four waves, WT_8 and WT_256 of eight), register-weight gemm_wr_kernel (WR) and k-grouped
// gemm_wk_kernel (WK).
enum MmId : int {
  MM_SMALL = 0, MM_WIDE = 1, MM_WIDE_D = 2, MM_BIG = 3, MM_WT = 4, MM_WR = 5, MM_WR_S = 6, MM_WR_M = 7, MM_WR_T = 8,
  MM_WR_3 = 9, MM_WT_8 = 10, MM_WT_256 = 11, MM_WK_GU4 = 12, MM_WK_GU6 = 13, MM_WK_GU8 = 14
};
// a workgroup's block of rows x 16-column weight tiles, and the k steps of one of its stages
struct MmInfo { int bm, bn_tiles, kss; };
constexpr MmInfo mm_info(int id) {
  switch (id) {
    case MM_WIDE: return {64, 16, 2};
    case MM_WIDE_D: return {64, 16, 2};
    case MM_BIG: return {128, 16, 2};
    case MM_WT: return {128, 12, 1};
    case MM_WT_8: return {128, 12, 1};
    case MM_WT_256: return {256, 12, 1};
    case MM_WR: return {128, 16, 1};
    case MM_WR_S: return {64, 8, 1};
    case MM_WR_M: return {128, 8, 1};
    case MM_WR_T: return {64, 4, 1};
    case MM_WR_3: return {128, 12, 1};
    case MM_WK_GU4: return {64, 6, 2};
    case MM_WK_GU6: return {96, 6, 2};
    case MM_WK_GU8: return {128, 6, 2};
    default: return {64, 8, 2};
  }
}

// rows from which the lm_head (with its confidence statistics) takes the register-weight kernel (us per
// launch with the statistics, fp16, register-weight / 64 x 256 LDS-staged blocks: 199 / 228-232 at 256 rows,
// 326 / 386 at 512, even at 112-128)
#ifndef FD_WR_LM_MIN_ROWS
#define FD_WR_LM_MIN_ROWS 256
#endif
// Rows from which a projection takes the register-weight kernel by default, where the counts in mm_choice have not
// decided before.  Measured (1.5B, us per
// launch, register-weight / previous kernel): gate_up 53 / 47 at 512 rows, 110 / 118 at 2048, 377 / 448
// at 8192; down 40 / 30, 79 / 80, 189 / 192; qkv 37 / 31 at 2048, 75 / 106 at 8192; o_proj 38 / 23,
// 57 / 70.  Below these sizes its 128 x 256 blocks leave too few workgroups without a k split.
inline int wr_default_min_rows(int cfg) {
  if (cfg == CFG_LM_HEAD) return FD_WR_LM_MIN_ROWS;
  return cfg == CFG_GATE_UP || cfg == CFG_DOWN ? 2048 : 4096;
}
// the blocks of an M-row launch on kernel id
inline int mm_blocks(int id, int M, int ntiles) {
  const MmInfo b = mm_info(id);
  return (M + b.bm - 1) / b.bm * ((ntiles + b.bn_tiles - 1) / b.bn_tiles);
}
// Whether wgs workgroups leave at most 7 of every 32 units of a round of `units` idle.  (The line lies between down of
// 3100 rows, 200 blocks of 128 x 192 on 256 units, 102.7 us against the LDS-staged 99.5, and of 2200 rows, 204 of
// 128 x 256, 77.3 against 92.3; gate_up of 896 x 4864, 390 blocks of 128 x 256 for 512, 34.3 against 29.8 at 1200 rows,
// 429 for 512, 34.6 against 39.2 at 1344.)
inline bool mm_fills(int wgs, int units) { return wgs <= units && 32 * wgs > 25 * units; }
// The most k splits, of at least 16 stages each, of nb blocks within one round of a workgroup per compute unit (0: the
// blocks alone are more).
inline int mm_round_split(int nb, int nst, const MmPolicy& pol) {
  int split = nb <= pol.cus ? 1 : 0;
  for (int d = 2; d <= 16 && nb * d <= pol.cus; ++d)
    if (nst % d == 0 && nst / d >= std::max(16, pol.min_stages)) split = d;
  return split;
}
// Down on register-weight 128 x 256 blocks whose splits come to one round: where they fill it, or, for weights
// that are no whole number of 192-column blocks (the LDS-staged 64 x 256 blocks take those below 2048 rows), take
// more than half of it (2048 x 5632, us: 53 against 67 at 1100 rows, 56 / 72 at 1700; 896 x 4864: 29 / 36, 32 / 40).
inline bool mm_down_round(int M, int ntiles, int ks, const MmPolicy& pol) {
  const int nb = mm_blocks(MM_WR, M, ntiles), wgs = nb * mm_round_split(nb, ks, pol);
  if (ntiles % 12 == 0) return mm_blocks(MM_WR_3, M, ntiles) <= pol.cus && mm_fills(wgs, pol.cus);
  return M < 2048 && 2 * wgs > pol.cus;
}
inline int mm_choice(int cfg, int M, int ntiles, int ks, const MmPolicy& pol) {
  // The large blocks by how their counts fill the compute units, us per launch at the 1.5B shapes.
  // gate_up on register-weight 128 x 256 where those are one round of two workgroups per unit (641 to 896 rows) / LDS-
  // staged: 50.7 / 56.7 at 660 rows, 51.7 / 59.4 at 896 (but 51.3 / 43.9 at 640, 68.3 / 59.1 at 900).  o_proj on
  // register-weight 128 x 192 once its 64 x 128 blocks pass two workgroups per unit (2688 rows) / 64 x 128: 28.6 / 36.0
  // at 2700, 28.8 / 36.7 at 3000 (28.9 / 24.1 at 2688).  Down, register-weight 128 x 192 where those fill a round /
  // LDS-staged: 31.6 / 33.1 at 660 rows (128 x 128 blocks, one and an eighth rounds: 42.2), 37.6 / 40.3 at 896, 39.4 / 41.3
  // at 1024, 55.5 / 52.5 at 1100, 59.9 / 59.4 at 1400, 61.7 / 64.1 at 1600, 101 / 97 at 2800, 98 / 105 at 3500; 128 x 256
  // where those do, 47.8 / 53.4 at 1200, 78.6 / 86.9 at 2100, 79.4 / 90.1 at 2400, 82.4 / 95.6 at 2688.
  if (pol.wr_min_rows == 0 && ((pol.wr_ops >> cfg) & 1) && pol.wr_ffn < 0) {
    const bool b3 = pol.wr3 && ntiles % 12 == 0;
    if (cfg == CFG_GATE_UP && M > 400 && mm_fills(mm_blocks(MM_WR, M, ntiles), 2 * pol.cus)) return MM_WR;
    if (cfg == CFG_OPROJ && b3 && mm_blocks(MM_SMALL, M, ntiles) > 2 * pol.cus) return MM_WR_3;
    if (cfg == CFG_DOWN && M > 640) {
      const int nb = mm_blocks(MM_WR_3, M, ntiles);
      if (b3 && mm_fills(nb * mm_round_split(nb, ks, pol), pol.cus)) return MM_WR_3;
      if (mm_down_round(M, ntiles, ks, pol)) return MM_WR;
      if (ntiles % 12 == 0 && M > 2048 && nb <= pol.cus) return MM_WT;
    }
  }
  const int min_rows = pol.wr_min_rows > 0 ? pol.wr_min_rows : wr_default_min_rows(cfg);
  if (M >= std::max(min_rows, 33) && ((pol.wr_ops >> cfg) & 1))
    return pol.wr3 && (cfg == CFG_OPROJ || cfg == CFG_DOWN) && ntiles % 12 == 0 ? MM_WR_3 : MM_WR;
  // qkv and o_proj below that: 64 x 128 register-weight blocks (us per launch, qkv including its norm pass,
  // against the LDS-staged 64 x 128 kernel): qkv 16.2 / 14.9 at 128 rows, 23.2 / 20.2 at 512, 26.2 / 19.4
  // at 1024, 30.8 / 28.6 at 2048; o_proj 15.2 / 14.0 at 384, 15.4 / 14.0 at 512, 19.3 / 15.1 at 1024, but
  // 23.3 / 26.4 at 2048 (equal below 384).  Up to 512 rows 64 x 64 blocks, twice the workgroups, do better
  // still (us, 64 x 128 / 64 x 64 blocks): qkv 14.4 / 13.4 at 128 rows, 15.7 / 13.7 at 256, 16.8 / 14.9 at
  // 512 (but 19.4 / 21.2 at 1024); o_proj 12.8 / 11.9, 12.8 / 11.9, 14.0 / 12.0 (15.1 / 21.4 at 1024)
  // o_proj while its 64 x 128 blocks are one round of the compute units (1344 rows: 16.1 / 20.0 at 1300, 25.9 / 23.3
  // at 1500; 896 columns, 2304 rows: 17.0 / 22.7 at 1800, 17.4 / 23.0 at 2300)
  if (M >= 33 && ((pol.wr_small_ops >> cfg) & 1) && (cfg == CFG_QKV || (cfg == CFG_OPROJ && mm_blocks(MM_WR_S, M, ntiles) <= pol.cus)))
    return M <= 512 ? MM_WR_T : MM_WR_S;
  // gate_up and down of short calls: register-weight blocks too (FDLLM_WR_FFN picks 64 x 128 or 128 x 128 blocks
  // below 1024 rows, or the LDS-staged kernels).
  if (M >= 33 && M < 1024 && pol.wr_ffn >= 0 && (cfg == CFG_GATE_UP || cfg == CFG_DOWN)) {
    const int sh = cfg == CFG_GATE_UP ? 0 : 1;
    if ((pol.wr_ffn >> sh) & 1) return MM_WR_S;
    if ((pol.wr_ffn >> (sh + 2)) & 1) return MM_WR_M;
  } else if (M >= 33 && cfg == CFG_GATE_UP) {
    // us per launch including its norm pass, k groups / 64 x 128 / 128 x 128 / LDS-staged blocks: 33 rows 17.5 /
    // 20.5, 64 rows 18.5 / 21.0 / 22.7, 96 rows 20.5 / - / 24.1, 128 rows 23.3 / 29.9 / 26.0, 129 rows 30.8 / 27.2 /
    // 31.6, 192 rows 32.5 / 28.8 / 34.2, 208 rows - / 34.5 / 35.0, 256 rows 37.6 / 37.5 / 37.1 / 43.2, 320 rows - / 37.8
    // / 34.9 / 41.7, 384 rows - / 43.2 / 36.6 / 42.1, 416 rows - / 44.3 / 43.0 / 42.0, 512 rows - / 54.1 / 48.8 / 42.6
    if (M <= 128) return M <= 64 ? MM_WK_GU4 : M <= 96 ? MM_WK_GU6 : MM_WK_GU8;
    if (M <= 224) return MM_WR_S;
    // (2048 x 11008, 519 blocks of 128 x 128 for two workgroups per unit: 53.7 / 51.7 LDS-staged at 300 rows)
    if (M <= 400 && mm_blocks(MM_WR_M, M, ntiles) <= 2 * pol.cus) return MM_WR_M;
  } else if (M >= 33 && cfg == CFG_DOWN) {
    // us per launch with its split sum, 64 x 128 blocks / LDS-staged: 64 rows 14.4 / 21.4, 128 rows 15.7 / 21.4, 192
    // rows 16.7 / 27.1, 256 rows 17.8 / 22.6, 320 rows 20.9 / 23.8, 352 rows 27.7 / 24.1.  From 417 to 640 rows
    // 128 x 128 blocks where their splits fill a round (or half of it, as in mm_down_round): in a prefill, us per layer
    // against the LDS-staged blocks: 448 rows 90.7 / 93.0, 509 rows 91.6 / 93.5, 576 rows 102.4 / 109.3, 640 rows 104.9 /
    // 111.3 (but 384 rows 95.4 / 88.5, 768 rows 126.3 / 120.6)
    if (M <= 320) return MM_WR_S;
    if (M > 416 && M <= 640) {
      const int nb = mm_blocks(MM_WR_M, M, ntiles), wgs = nb * mm_round_split(nb, ks, pol);
      if (ntiles % 12 == 0 ? mm_fills(wgs, pol.cus) : 2 * wgs > pol.cus) return MM_WR_M;
    }
  }
  switch (cfg) {
    case CFG_LM_HEAD: return MM_WIDE;  // one 256-column confidence tile per block column
    case CFG_GATE_UP:
      if (M > 256 && M <= pol.wt256 && ntiles % 12 == 0) return MM_WT_256;
      if (M >= 256 && ntiles % 12 == 0) return (pol.wt8 & 1) ? MM_WT_8 : MM_WT;
      return M >= 1024 ? MM_BIG : MM_WIDE;
    case CFG_DOWN:
      if (M >= 256 && ntiles % 12 == 0) return (pol.wt8 & 2) ? MM_WT_8 : MM_WT;
      return M >= 1024 ? MM_WIDE_D : MM_SMALL;
    default:  // qkv, o_proj: the LDS-staged kernel measured slower at their widths (2048 / 1536 columns)
      return MM_SMALL;
  }
}

// The k splits of an M-row launch on kernel id over nst stages: 1 unless it leaves compute units idle.
inline int mm_split(int cfg, int id, int M, int ntiles, int nst, const MmPolicy& pol) {
  const int wgs = mm_blocks(id, M, ntiles);
  // k split: the smallest divisor of the stage count that brings the launch to mm_target_wgs
  // workgroups (at most 8 splits of at least mm_min_stages stages), else the largest such divisor
  // (up to 128 rows, half the target: a split's fp32 partials and its epilogue launch cost more
  // than the idle compute units; measured on the 128-row batched step, 3.15 -> 2.93 ms)
  // o_proj (48 k steps) a quarter: at 512 rows its 96 workgroups without a split took 15.4 us against
  // 18.9 us split three ways with the epilogue launch
  int target = M <= 128 ? pol.target_wgs / 2 : pol.target_wgs;
  if (cfg == CFG_OPROJ) target /= 4;
  // qkv on the 64 x 128 (and 64 x 64) register-weight blocks half: 17.1 against 20.4 us at 512 rows (128 workgroups
  // without a split against 256 with one), 13.8 against 14.5 at 128 (two splits against four)
  if (cfg == CFG_QKV && (id == MM_WR_S || id == MM_WR_T)) target /= 2;
  // down above 128 rows seven eighths: at 512 rows seven splits (224 workgroups) against eight (256)
  // measured 3.92 against 3.94-3.95 ms per batched step (fewer partials for the split sum; five
  // splits 4.03, ten 3.95)
  if (cfg == CFG_DOWN && M > 128) target = target * 7 / 8;
  if (id == MM_WT_256 || (id >= MM_WK_GU4 && id <= MM_WK_GU8)) target = 0;  // no split
  int split = 1;
  const int max_split = id == MM_WR || id == MM_WR_S || id == MM_WR_M || id == MM_WR_T || id == MM_WR_3 ? 16 : 8;
  if (pol.force_split > 1 && cfg != CFG_LM_HEAD && nst % pol.force_split == 0 && nst / pol.force_split >= pol.min_stages)
    split = pol.force_split;
  else
    for (int d = 2; d <= max_split && wgs * split < target && cfg != CFG_LM_HEAD; ++d)
      if (nst % d == 0 && nst / d >= pol.min_stages) split = d;
  // (at 1152 rows five splits of 54 blocks took 58.9 us, at 1200 four of 60 blocks 47.8)
  if (cfg == CFG_DOWN && id == MM_WR && pol.wr_min_rows == 0 && pol.force_split <= 1 && pol.target_wgs >= pol.cus &&
      mm_down_round(M, ntiles, nst, pol))
    split = mm_round_split(wgs, nst, pol);
  if (cfg == CFG_DOWN && id == MM_WR_S && pol.wr_ffn < 0 && pol.force_split <= 1 && pol.target_wgs >= pol.cus) {
    // down's 64 x 128 blocks: the most splits up to seven that leave every XCD a workgroup per compute unit
    // at most (us per launch with its split sum; 130 rows: 5 splits 16.7, 7 splits 21.5, of 35 workgroups on
    // seven XCDs; 64 rows: 7 splits 14.4, 8 splits 14.7, 14 splits 16.8, whose partials cost more than their workgroups
    // give).  Eight where none of five to seven divides the stages and four leave over half the units without a
    // workgroup or more than 64 stages each (four / eight: 2048 x 11008 64 rows 26.8 / 19.5, 128 rows 26.7 / 20.3, 896 x
    // 4864 40 rows 12.7 / 11.1; but 2048 x 5632 128 rows 14.0 / 14.6).
    const int fit = std::min(8, std::max(1, pol.target_wgs / 8 / ((wgs + 7) / 8)));
    split = 1;
    for (int d = 2; d <= fit; ++d)
      if (nst % d == 0 && nst / d >= pol.min_stages &&
          (d < 8 || (split < 5 && (2 * wgs * split < pol.cus || nst / split > 64))))
        split = d;
  }
  return split;
}

}  // namespace fdllm
