// Number of activation buffers of the mid-batch kernel, shared by its launcher and by what reports it.
#pragma once

namespace matgptq {

// Whether a walk over K (skinny_gfx950.hip) takes two activation buffers: on pre-sliced codes and up to 32 batch rows per
// workgroup (the second buffer is another 32 KB per 16 batch rows).  `r`: row blocks and `mb`: blocks of 16 batch rows of a
// workgroup; a wave walks ceil(k_tiles / 8) tiles.  What two buffers gain is the wait of a wave for its next tile, and in an odd walk
// the empty tile that the loop of pairs ends with; what they cost is registers (two sets of codes stay live) and, over
// 64 KB, the second workgroup of a CU.  One against two buffers on some 15000 random calls (M = 5..128, K = 256..8192, all bitwidths,
// groups and storage types; mean gain, share that lost more than 1.5 %):
//  * walks of one tile have nothing to fetch ahead: one buffer and one register set, the next workgroup of the CU instead
//    (1.07 to 1.14 times faster than with two, planes 1.18 to 1.25, over 10300 random calls of 5 to 96 batch rows, none slower);
//  * one row block and 16 batch rows: two or three tiles 6.7 %, 0.1 %; longer walks 5 %, 1 % (4096 x 4096 at M = 12:
//    5.53 -> 5.28 us) without group 32 with zero points (0 to 2 %, 7 %: four scales and zeros per tile in two sets) and
//    without even walks at 6 bits (2.5 %, 17 %);
//  * one row block and 32 batch rows: three tiles 7.7 %, none; two 9.6 %, 0.5 %, those in more workgroups than CUs
//    (4544 x 1920 at M = 26, 8 bits: 8.37 -> 8.78 us); odd walks of fp16 storage 3 to 5 %, none.  Not the others
//    (even walks from four tiles on bf16 lose 1 %, half of them; 1 to 3 % on fp16 with 9 % that lose; odd ones on bf16 1 to 4 %, 6 %);
//  * two or four row blocks, 16 batch rows and more workgroups than CUs, fp16 storage: 6.6 %, 0.2 % (28672 x 4096 at M = 12:
//    17.6 -> 16.0 us) without four row blocks at 6 bits with zero points (0 %, a third; 56960 x 2816 at M = 15: 31.4 -> 35.4 us) and
//    8 bits at group 32 (16384 x 2048 at M = 12 11.2 against 12.3); bf16 storage forms its weights in fp32 and takes more
//    registers (28672 x 4096 at M = 13 17.3 against 19.3).
// Elsewhere one buffer is as fast or ahead by up to 5 % (8192 x 3584 at M = 16: 6.74 against 7.02 us).
inline bool midbatch_two_buffers(int bits, bool bf16, int group_size, bool zeros, int r, int mb, bool master, int k_tiles,
                                 int M, int row_blocks) {
  if (master || r > 4 || mb > 2) return false;
  const int walk = (k_tiles + 7) / 8;
  const int workgroups = ((row_blocks + r - 1) / r) * ((M + 16 * mb - 1) / (16 * mb));
  if (walk <= 1) return false;
  if (r > 1)
    return mb == 1 && !bf16 && workgroups > 256 && !(group_size == 32 && bits == 8) && !(r == 4 && bits == 6 && zeros);
  if (M > 32 && k_tiles > 32) return false;  // (several blocks of batch rows and a long walk)
  const bool odd = walk % 2 != 0;
  if (mb == 1) return walk <= 3 || (!(group_size == 32 && zeros) && (odd || bits != 6));
  return walk == 3 || (walk == 2 && workgroups <= 256) || (odd && !bf16);
}

}  // namespace matgptq
