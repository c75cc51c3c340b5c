// When the few-rows kernel (fewrows_gfx950.hip) runs and with how many row blocks per workgroup, shared by the entry points,
// the launcher and what reports it.
#pragma once

namespace matgptq {

constexpr int kFewRowsMaxM = 16;
constexpr int kFewRowsWaves = 8;

// Row blocks of 16 weight rows per workgroup (1, 2 or 4) for M batch rows, or 0: another kernel takes the call.
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
inline int few_rows_row_blocks(int bits, int group_size, bool bf16, bool master, int M, int row_blocks, int k_tiles) {
  if (group_size == 32 || M > kFewRowsMaxM) return 0;
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

}  // namespace matgptq
