// When the few-rows kernel (fewrows_gfx950.hip) runs and with how many row blocks per workgroup, shared by the entry points,
// the launcher and what reports it.
#pragma once

namespace matgptq {

constexpr int kFewRowsMaxM = 64;
constexpr int kFewRowsWaves = 8;

// Workgroup of the few-rows kernel: row blocks of 16 weight rows (0: another kernel takes the call) and batch rows, 16 (of
// which fewer are held where M is 4 or 8 at most) or 32.
struct FewRows {
  int row_blocks, batch_rows;
};

// Batch rows that a workgroup really holds for a call of M.
constexpr int few_rows_held(FewRows f, int M) { return M <= 4 ? 4 : M <= 8 ? 8 : f.batch_rows; }

// Most row blocks of 16 weight rows per workgroup that the registers hold, by the format and the batch rows per workgroup.
constexpr int few_rows_most_row_blocks(int bits, bool master, int rows) {
  if (bits > (master ? 4 : 6)) return 2;
  return rows > 16 && bits <= 4 && !master ? 8 : 4;
}

// Where the lines of both rules lie: some 90000 random calls (every bitwidth and storage type, group sizes 128 and -1, 64 to 65536
// weight rows, K = 128 to 28672, weights from HBM) against the kernel that runs without the rule.  Geometric mean of the speed-up and
// share of calls that lost more than 2 % (profiles/fewrows_random_calls.txt has the table of what is left).
//
// Seventeen to 64 batch rows: the smallest workgroup whose count does not exceed the CUs.  The activations are copied once per
// workgroup column and the codes' masks and ORs are paid once per block of batch rows, so larger workgroups spend less, but two
// workgroups of a CU halve each other's rate while a CU without one halves the chip's.
//  * walks of one tile, whose workgroups are short and up to four to a CU: 16 x 16 up to 768 workgroups, two row blocks up to 1536
//    from four K tiles (1.5, none).  Not 641 to 1024 of seven or eight tiles, one round of the mid-batch kernel's workgroups of two
//    row blocks (1.04, but 0.85 to 0.95 on a third), and not past 560 of a single K tile on fp16 storage (0.98, half);
//  * 17 to 32 rows: 16 x 16 up to 128 row blocks (1.2 to 1.4, none), two row blocks of 16 up to 256 from walks of four tiles (1.19,
//    none), two of 32 (to 512) from walks of three (1.25, none; of two 0.95), four of 32 (to 1024) 1.23, none; beyond as many as the
//    format holds: eight 1.2, none, from walks of three (past 2048 row blocks of four; three 1.02, a quarter), four, at 6 bits, from
//    walks of four (1.13, 5 %; three 1.0, half);
//  * 33 to 48 rows: 16 x 16 (to 85 row blocks) 1.25, none; two of 16 (129 to 170) and four of 16 (257 to 340) 1.6, none; between
//    these lines 0.9 to 1.05: nothing;
//  * 49 to 64 rows: 16 x 16 (to 64) from walks of three 1.38, none; two of 32 on walks of three 1.24, none; four of 32 (257 to
//    512) on walks of two to five tiles, and longer ones of bf16 storage, 1.2, none; elsewhere 0.9 to 1.02: nothing.
// On planes the same lines hold (1.2 to 1.6), but for two row blocks of 16 at 6 and 8 bits (0.74 to 1).
// fp16 storage with a scale per tile is not taken from 32 rows on.  That is a choice, not a measurement: those calls keep the
// results they have always had.  No property of the results rests on it: shorter batches of the same layer multiply unrounded
// weights here, and longer ones add in other orders, tile by tile, half by half or in eighths.
inline FewRows few_rows_mid(int bits, int group_size, bool bf16, bool master, int M, int row_blocks, int k_tiles) {
  const FewRows none{0, 0};
  if (!bf16 && group_size == 128 && M >= 32) return none;
  const int walk = (k_tiles + kFewRowsWaves - 1) / kFewRowsWaves;
  auto fits = [&](int r, int rows) {
    return r <= few_rows_most_row_blocks(bits, master, rows) && (row_blocks + r - 1) / r * ((M + rows - 1) / rows) <= 256;
  };
  const int blocks = row_blocks * ((M + 15) / 16);
  if (walk == 1 && k_tiles >= 7 && blocks > 640 && blocks <= 1024) return none;
  if (k_tiles == 1 && !bf16 && !master && blocks > 560) return none;
  if (walk == 1) return blocks <= 768 ? FewRows{1, 16} : blocks <= 1536 && k_tiles >= 4 ? FewRows{2, 16} : none;
  if (fits(1, 16)) return M > 48 && walk == 2 ? none : FewRows{1, 16};
  if (M <= 32) {
    if (fits(2, 16)) return walk >= 4 && !(master && bits > 4) ? FewRows{2, 16} : none;
    if (fits(2, 32)) return walk >= 3 ? FewRows{2, 32} : none;
    if (fits(4, 32)) return {4, 32};
    const int most = few_rows_most_row_blocks(bits, master, 32);
    if (master || most < 4 || row_blocks <= 1024 || walk < (most == 4 || row_blocks > 2048 ? 4 : 3)) return none;
    return bf16 || most == 4 || row_blocks <= 2048 ? FewRows{most, 32} : none;
  }
  if (M <= 48) {
    if (row_blocks > 128 && fits(2, 16)) return {2, 16};
    return row_blocks > 256 && fits(4, 16) ? FewRows{4, 16} : none;
  }
  if (walk == 3 && !fits(2, 16) && fits(2, 32)) return {2, 32};
  return row_blocks > 256 && (bf16 || walk <= 5) && fits(4, 32) ? FewRows{4, 32} : none;
}

// One to sixteen batch rows: row blocks of 16 weight rows per workgroup (1, 2 or 4), or 0.
// `master`: the codes are master-resident planes.
//  * five to sixteen rows: everywhere (1.18, 0.4 %; planes 1.23, 0.6 %) but for 8 bits on fp16 storage on more than 2500 row blocks
//    of one or two K tiles, where the decode kernel's workgroups of 16 row blocks pay their start less often (0.78 to 0.95); group
//    size 32 has a scale per octet, which takes the fold four times per tile: not built;
//  * three and four rows (1.19, 2 %; planes 1.25, 1 %): not where the gemv kernel's sixteen waves with four tiles in flight each hide
//    more of the latency, on walks past 60 tiles of up to 256 row blocks (0.95) and past 56 (planes 60) of up to 512 with two per
//    workgroup (0.95 to 1.03, a third to a half), nor on many row blocks of 9 to 16 tiles, of which half of the waves walk one and
//    half two (from 1500 row blocks 0.9 to 1.07; planes from 2200 0.98), or up to 8 on more than 3000 at one scale per row (1.03, a
//    third);
//  * one and two rows, where the gemv kernel's staging is cheap: short walks on few row blocks (1.03 and 1.07, planes 1.1 and 1.15;
//    one row past eight tiles 0.95 to 1.02), and planes of large layers, whose slice in registers two waves per SIMD more hide
//    (1.05 to 1.3; walks of 41 to 50 tiles 0.9 to 1.05);
//  * row blocks per workgroup: one while that fills the CUs, then as many as leave about 160 workgroups (512 row blocks at
//    M = 16: two row blocks 1.11, four 0.96; 900: two 1.10, four 1.20).
inline int few_rows_small(int bits, int group_size, bool bf16, bool master, int M, int row_blocks, int k_tiles) {
  // (up to four rows of what the gemv kernel takes with the operator in front fused into it stay there, so that a layer gives
  // the same bits with and without that)
  if (M <= 4 && !bf16 && !master && group_size == 128) return 0;
  if (M == 1) {
    if (master)
      return (k_tiles <= 16 && row_blocks <= 600) || (k_tiles <= 24 && row_blocks <= 256) ||
                     (k_tiles > 50 && k_tiles <= 64 && row_blocks > 1024) ? 1 : 0;
    return k_tiles <= 8 && row_blocks <= (k_tiles > 4 ? 512 : 256) ? 1 : 0;
  }
  if (M == 2) {
    if (master)
      return (k_tiles <= 24 && row_blocks <= 600) || (k_tiles <= 8 && row_blocks <= 1024) ||
                     (k_tiles > 50 && k_tiles <= 120 && row_blocks > 800) ? 1 : 0;
    return (k_tiles <= 24 && row_blocks <= 400) || (k_tiles <= 8 && row_blocks <= 640) ? 1 : 0;
  }
  if (M <= 4) {
    if (row_blocks <= 256 && k_tiles > 60) return 0;
    if (row_blocks >= 320 && row_blocks <= 512 && k_tiles > (master ? 60 : 56)) return 0;
    if (row_blocks > (master ? 2200 : 1500) && k_tiles > 8 && k_tiles <= 16) return 0;
    if (group_size == -1 && !master && row_blocks > 3000 && k_tiles <= 8) return 0;
    return row_blocks < 320 ? 1 : 2;
  }
  if (bits == 8 && !bf16 && !master && row_blocks > 2500 && k_tiles <= 2) return 0;
  if (M <= 8 && row_blocks <= 512) return row_blocks < 320 ? 1 : 2;
  for (int r = bits > (master ? 4 : 6) ? 2 : 4; r > 1; r >>= 1)
    if ((row_blocks + r - 1) / r >= 160) return r;
  return 1;
}

// The instantiations that the two rules can ask for (and no others are built): `held` as few_rows_held gives it, `one`: walks of
// one tile.
constexpr bool few_rows_built(int bits, int group_size, bool bf16, bool master, int r, int held, bool one) {
  if (held == 32) return !one && r >= 2 && r <= few_rows_most_row_blocks(bits, master, 32);
  if (held == 4) return r <= 2 && (bf16 || master || group_size != 128);
  return r <= 4 && r <= few_rows_most_row_blocks(bits, master, 16);
}

// The workgroup for M batch rows.  `master`: the codes are master-resident planes.
inline FewRows few_rows(int bits, int group_size, bool bf16, bool master, int M, int row_blocks, int k_tiles) {
  if (group_size == 32 || M > kFewRowsMaxM) return {0, 0};
  if (M > 16) return few_rows_mid(bits, group_size, bf16, master, M, row_blocks, k_tiles);
  return {few_rows_small(bits, group_size, bf16, master, M, row_blocks, k_tiles), 16};
}

}  // namespace matgptq
