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

// Seventeen to 64 batch rows.
// The smallest workgroup whose count does not exceed the CUs: the activations are copied once per workgroup column and the
// codes' masks and ORs are paid once per block of batch rows, so larger workgroups spend less, but two workgroups of a CU halve
// each other's rate while a CU without one halves the chip's.  Some 7000 random calls against what ran there before
// (mid-batch kernel, some 64 x 128 tiles), geometric mean and share that lost more than 2 %:
//  * walks of one tile, whose workgroups are short and up to four to a CU: 16 x 16 up to 768 workgroups 1.4 to 1.9, 2 %; two
//    row blocks up to 1536 from four K tiles 1.12 to 1.36, 8 % (16 x 16 there 1.06 to 1.24); beyond 0.85 to 1.1.  Not 641 to 1024 of
//    seven or eight tiles, one round of the mid-batch kernel's workgroups of two row blocks (1.04, but 0.85 to 0.95 on a third);
//  * 17 to 32 rows: 16 x 16 (up to 128 row blocks) 1.12 to 1.29, 1 %; two row blocks of 16 (to 256) from walks of four
//    tiles 1.05 to 1.1, 15 % (of three 1.01, 25 %; of two 0.95); two of 32 (to 512) from walks of three 1.18, 1 % (of two
//    1.03, 42 %); four of 32 (to 1024) 1.2, none; eight of 32 (beyond) 1.21, 1 % from walks of three (of two 0.98);
//  * 33 to 48 rows, where the mid-batch kernel multiplies 64: 16 x 16 (to 85 row blocks) 1.05 to 1.12, 5 %; two of 16 (129 to
//    170) 1.3; four of 16 (257 to 340) 1.35, 1 %; between these lines 0.9 to 1.05: nothing;
//  * 49 to 64 rows: 16 x 16 (to 64) from walks of three 1.12, 12 % (of two 1.06, a third); 32 batch rows on walks of three
//    tiles 1.13, 13 %; four of 32 (257 to 512) on walks of two to five tiles, and longer ones of bf16 storage, 1.1, 10 %;
//    elsewhere 0.9 to 1.02: nothing.
// On planes the same lines hold (1.18, 1.29 and 1.29 over all of the three ranges of M), but for two row blocks of 16 at 6 and 8
// bits (0.74 to 1).
// fp16 storage with a scale per tile stays with the kernels that form weights from 32 rows on: a prompt's results do not move
// with the way it is split into calls.
inline FewRows few_rows_mid(int bits, int group_size, bool bf16, bool master, int M, int row_blocks, int k_tiles) {
  const FewRows none{0, 0};
  if (!bf16 && group_size == 128 && M >= 32) return none;
  const int walk = (k_tiles + kFewRowsWaves - 1) / kFewRowsWaves;
  auto fits = [&](int r, int rows) {
    return r <= few_rows_most_row_blocks(bits, master, rows) && (row_blocks + r - 1) / r * ((M + rows - 1) / rows) <= 256;
  };
  const int blocks = row_blocks * ((M + 15) / 16);
  if (walk == 1 && k_tiles >= 7 && blocks > 640 && blocks <= 1024) return none;
  if (walk == 1) return blocks <= 768 ? FewRows{1, 16} : blocks <= 1536 && k_tiles >= 4 ? FewRows{2, 16} : none;
  if (fits(1, 16)) return M > 48 && walk == 2 ? none : FewRows{1, 16};
  if (M <= 32) {
    if (fits(2, 16)) return walk >= 4 && !(master && bits > 4) ? FewRows{2, 16} : none;
    if (fits(2, 32)) return walk >= 3 ? FewRows{2, 32} : none;
    if (fits(4, 32)) return {4, 32};
    const int most = few_rows_most_row_blocks(bits, master, 32);
    return !master && most >= 4 && row_blocks > 1024 && walk >= 3 && (bf16 || most == 4 || row_blocks <= 2048) ? FewRows{most, 32} : none;
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
// Where the lines lie (some 30000 random calls against what ran there before; geometric means of the speed-up):
//  * five to sixteen rows: everywhere (1.08 to 1.6, the larger the shorter the walk); group size 32 has a scale per octet,
//    which takes the fold four times per tile: not built;
//  * three and four rows (1.05 to 1.4): not on long walks over few row blocks, where the gemv kernel's sixteen waves with four
//    tiles in flight each hide more of the latency (4096 x 14336: 0.95);
//  * one and two rows, where the gemv kernel's staging is cheap: short walks on few row blocks (1.03 to 1.18), and planes of
//    large layers, whose slice in registers two waves per SIMD more hide (1.05 to 1.3); elsewhere 0.85 to 1.02;
//  * row blocks per workgroup: one while that fills the CUs, then as many as leave about 160 workgroups (512 row blocks at
//    M = 16: two row blocks 1.11, four 0.96; 900: two 1.10, four 1.20).
inline int few_rows_small(int bits, int group_size, bool bf16, bool master, int M, int row_blocks, int k_tiles) {
  // (up to four rows of what the gemv kernel takes with the operator in front fused into it stay there, so that a layer gives
  // the same bits with and without that)
  if (M <= 4 && !bf16 && !master && group_size == 128) return 0;
  if (M <= 2) {
    const bool short_walk = M == 1 ? k_tiles <= (master ? 24 : 16) && row_blocks <= 600
                                   : (k_tiles <= 24 && row_blocks <= (master ? 600 : 400)) || (k_tiles <= 8 && row_blocks <= 1024);
    const bool large_planes = master && k_tiles > 40 && row_blocks > (M == 1 ? 1024 : 600);
    return short_walk || large_planes ? 1 : 0;
  }
  if (M <= 4) {
    if (row_blocks <= 256 && k_tiles > 64) return 0;
    return row_blocks < 320 ? 1 : 2;
  }
  if (M <= 8 && row_blocks <= 512) return row_blocks < 320 ? 1 : 2;
  for (int r = bits > (master ? 4 : 6) ? 2 : 4; r > 1; r >>= 1)
    if ((row_blocks + r - 1) / r >= 160) return r;
  return 1;
}

// The workgroup for M batch rows.  `master`: the codes are master-resident planes.
inline FewRows few_rows(int bits, int group_size, bool bf16, bool master, int M, int row_blocks, int k_tiles) {
  if (group_size == 32 || M > kFewRowsMaxM) return {0, 0};
  if (M > 16) return few_rows_mid(bits, group_size, bf16, master, M, row_blocks, k_tiles);
  return {few_rows_small(bits, group_size, bf16, master, M, row_blocks, k_tiles), 16};
}

}  // namespace matgptq
