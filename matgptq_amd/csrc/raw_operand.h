// Codes as matrix operands without dequantisation: a pair of codes becomes a pair of storage-type numbers
// (fp16 or bf16) base + c by a mask and an OR, where `base` depends on the position of the field only.
// A product with them is corrected afterwards by  base + 2^(b-1)  times the sum of the activations, and
// scale and zero point are applied to the product of a whole group.
//
// fp16: with the exponent of 2^(10 - p) a mantissa step is 2^-p, so a field that starts at bit p of the
// half word reads as  2^(10 - p) + c  exactly, whatever p is: the field needs no shift of its own and the
// activations no scaling.  The higher the field, the smaller `base` and what cancels against it: sums keep
// their rounding errors at that of a small number (nibbles at bits 2 and 6 instead of 0 and 4 cost one shift
// per octet and take 3-bit sums of 128 columns from 5e-5 to 1e-5 of their size).  bf16 has 7 mantissa
// bits: 2^(7 - p) + c as long as the field ends at bit 6; fields that do not are shifted down first, and bytes
// are converted (c itself, base 0).
#pragma once
#include "tile_format.h"

namespace matgptq {

// two equal 16-bit numbers 2^e of the storage type
constexpr uint32_t pow2_pair(int e) {
  const uint32_t h = kBf16 ? (uint32_t)(127 + e) << 7 : (uint32_t)(15 + e) << 10;
  return h | (h << 16);
}
// bits of the small integer v (exact in either storage type), v > 0
constexpr uint32_t int_bits(int v) {
  int e = 0;
  while ((v >> (e + 1)) != 0) e++;
  return kBf16 ? ((uint32_t)(127 + e) << 7) | ((uint32_t)(v << (7 - (e < 7 ? e : 7))) & 0x7fu)
               : ((uint32_t)(15 + e) << 10) | ((uint32_t)(v << (10 - e)) & 0x3ffu);
}

template <int BITS, bool MASTER>
struct RawOperand {
  using Fmt = TileFormat<BITS, MASTER>;
  static constexpr bool kNibbles = BITS == 3 || BITS == 4 || (MASTER && BITS == 2);
  static constexpr int kMant = kBf16 ? 7 : 10;
  // position of pair i's field in octet j where it is masked
  static constexpr int pos(int j, int i) {
    if (BITS == 8 || (MASTER && BITS == 6)) return 0;
    if (kNibbles) return !kBf16 ? ((i & 1) ? 6 : 2) : BITS == 4 ? 0 : (i & 1) ? 4 : 0;
    if (BITS == 6) return kBf16 ? 0 : (i & 1) ? 4 : 0;
    if (kBf16) return Codec<2>::raw_shift(j, i);
    return (j & 1) == 0 ? ((i & 1) ? 6 : 4) : i == 0 || i == 3 ? 8 : i == 1 ? 4 : 6;  // 2 bits
  }
  static constexpr bool kBytes = kBf16 && BITS == 8;  // converted, base 0
  static constexpr int base(int j, int i) { return kBytes ? 0 : 1 << (kMant - pos(j, i)); }
  // (negative) operand pair that takes base and 2^(b-1) off again
  static constexpr uint32_t centre_pair(int j, int i) {
    const uint32_t h = int_bits(base(j, i) + (1 << (BITS - 1))) | 0x8000u;
    return h | (h << 16);
  }
  static constexpr bool kOddOctets = BITS == 2 && !MASTER;  // odd octets have other positions than even ones

  uint32_t g[3];  // VGPRs: pairs of 2^(kMant - p) for the positions in use, lowest first
  uint32_t m[4];  // SGPRs: field masks
  __device__ __forceinline__ RawOperand() {
    m[3] = 0;
    if constexpr (kNibbles) {
      g[0] = opaque_vgpr(pow2_pair(kMant - pos(0, 0)));
      g[1] = opaque_vgpr(pow2_pair(kMant - pos(0, 1)));
      g[2] = 0;
      m[0] = opaque_sgpr(kBf16 ? 0x000F000Fu : 0x003C003Cu);
      m[1] = opaque_sgpr(kBf16 ? 0x00F000F0u : 0x03C003C0u);
      m[2] = opaque_sgpr(0x44444444u);
    } else if constexpr (BITS == 2) {
      constexpr int low = kBf16 ? 0 : 4;
      for (int i = 0; i < 3; i++) {
        g[i] = opaque_vgpr(pow2_pair(kMant - low - 2 * i));
        m[i] = opaque_sgpr(0x00030003u << (low + 2 * i));
      }
    } else {
      g[0] = opaque_vgpr(pow2_pair(kMant));
      g[1] = opaque_vgpr(pow2_pair(kMant - 4));
      g[2] = 0;
      m[0] = opaque_sgpr(0x00030003u); m[1] = opaque_sgpr(0x00300030u);
      m[2] = opaque_sgpr(0x003C003Cu); m[3] = opaque_sgpr(0x03C003C0u);
    }
  }

  // the four pairs of octet J
  template <int J>
  __device__ __forceinline__ void octet(const uint32_t (&w)[Fmt::kWords], uint32_t (&r)[4]) const {
    if constexpr (kNibbles) {
      uint32_t x;
      if constexpr (MASTER) {
        x = master_nibble_word<BITS, J>(w);
      } else if constexpr (BITS == 4) {
        x = w[J];
      } else {
        const uint32_t low = (w[J >> 1] >> (2 * (J & 1))) & 0x33333333u;
        const uint32_t c = w[2];
        x = and_or(J == 0 ? (c << 2) : J == 1 ? (c << 1) : J == 2 ? c : (c >> 1), m[2], low);
      }
      if constexpr (kBf16 && BITS == 4) {  // a nibble at bit 4 would reach into the exponent
        r[0] = and_or(x, m[0], g[0]);
        r[1] = and_or(x >> 4, m[0], g[0]);
        r[2] = and_or(x >> 8, m[0], g[0]);
        r[3] = and_or(x >> 12, m[0], g[0]);
      } else {
        const uint32_t a = kBf16 ? x : x << 2, b = x >> (kBf16 ? 8 : 6);
        r[0] = and_or(a, m[0], g[0]);
        r[1] = and_or(a, m[1], g[1]);
        r[2] = and_or(b, m[0], g[0]);
        r[3] = and_or(b, m[1], g[1]);
      }
    } else if constexpr (BITS == 2) {
      // sixteen fields of two bits, field f of each half word at bit 2f; octet 2d holds fields 0..3, octet 2d + 1 fields 4..7
      const uint32_t x = w[J >> 1];
      const uint32_t x6 = x >> 6;
      if constexpr (kBf16) {
        if constexpr ((J & 1) == 0) {
          r[0] = and_or(x, m[0], g[0]);
          r[1] = and_or(x, m[1], g[1]);
          r[2] = and_or(x, m[2], g[2]);
          r[3] = and_or(x6, m[0], g[0]);
        } else {
          const uint32_t x12 = x >> 12;
          r[0] = and_or(x6, m[1], g[1]);
          r[1] = and_or(x6, m[2], g[2]);
          r[2] = and_or(x12, m[0], g[0]);
          r[3] = and_or(x12, m[1], g[1]);
        }
      } else {
        if constexpr ((J & 1) == 0) {
          const uint32_t up = x << 4;
          r[0] = and_or(up, m[0], g[0]);
          r[1] = and_or(up, m[1], g[1]);
          r[2] = and_or(x, m[0], g[0]);
          r[3] = and_or(x, m[1], g[1]);
        } else {
          r[0] = and_or(x, m[2], g[2]);
          r[1] = and_or(x6, m[0], g[0]);
          r[2] = and_or(x6, m[1], g[1]);
          r[3] = and_or(x6, m[2], g[2]);
        }
      }
    } else if constexpr (BITS == 6 && !MASTER) {
      const uint32_t h = w[J], l = (J & 1) ? (w[4 + (J >> 1)] >> 8) : w[4 + (J >> 1)];
      if constexpr (kBf16) {  // six bits at bit 4 would reach into the exponent
        r[0] = and_or(h << 2, m[2], opaque_vgpr(and_or(l, m[0], g[0])));
        r[1] = and_or(h >> 2, m[2], opaque_vgpr(and_or(l >> 4, m[0], g[0])));
        r[2] = and_or(h >> 6, m[2], opaque_vgpr(and_or(l >> 2, m[0], g[0])));
        r[3] = and_or(h >> 10, m[2], opaque_vgpr(and_or(l >> 6, m[0], g[0])));
      } else {
        const uint32_t hs = h << 2, hs6 = h >> 6, l2 = l >> 2;
        // (the inner result is hidden from the optimiser, which would regroup the two instructions)
        r[0] = and_or(hs, m[2], opaque_vgpr(and_or(l, m[0], g[0])));
        r[1] = and_or(hs, m[3], opaque_vgpr(and_or(l, m[1], g[1])));
        r[2] = and_or(hs6, m[2], opaque_vgpr(and_or(l2, m[0], g[0])));
        r[3] = and_or(hs6, m[3], opaque_vgpr(and_or(l2, m[1], g[1])));
      }
    } else {
      // bytes.  Pre-sliced: pairs 2d, 2d + 1 = bytes (0, 2) and (1, 3) of word 2J + d; planes: pair i = bytes i / 2 and
      // i / 2 + 2 of byte word i % 2
      uint32_t a, b;
      if constexpr (MASTER) {
        a = master_byte_word<BITS, J, 0>(w);
        b = master_byte_word<BITS, J, 1>(w);
      } else {
        a = w[2 * J];
        b = w[2 * J + 1];
      }
      const uint32_t p0 = a, p1 = MASTER ? b : a, p2 = MASTER ? a : b, p3 = b;
      if constexpr (kBf16 && BITS == 8) {
        r[0] = bytes_bf16<0>(p0);
        r[1] = bytes_bf16<MASTER ? 0 : 1>(p1);
        r[2] = bytes_bf16<MASTER ? 1 : 0>(p2);
        r[3] = bytes_bf16<1>(p3);
      } else if constexpr (kBf16) {  // six bits: 128 + c
        constexpr uint32_t fill = 0x43434343u;
        r[0] = __builtin_amdgcn_perm(fill, p0, 0x04020400u);
        r[1] = __builtin_amdgcn_perm(fill, p1, 0x04020400u);
        r[2] = __builtin_amdgcn_perm(fill, p2, 0x04030401u);
        r[3] = __builtin_amdgcn_perm(fill, p3, 0x04030401u);
      } else {
        constexpr uint32_t fill = 0x64646464u;
        r[0] = __builtin_amdgcn_perm(fill, p0, 0x04020400u);
        r[1] = __builtin_amdgcn_perm(fill, p1, MASTER ? 0x04020400u : 0x04030401u);
        r[2] = __builtin_amdgcn_perm(fill, p2, MASTER ? 0x04030401u : 0x04020400u);
        r[3] = __builtin_amdgcn_perm(fill, p3, 0x04030401u);
      }
    }
  }

  // bytes B and B + 2 as bf16: eight significant bits, so the upper half of the fp32 number is exact
  template <int B>
  __device__ __forceinline__ static uint32_t bytes_bf16(uint32_t x) {
    const float a = (float)((x >> (8 * B)) & 0xffu), b = (float)((x >> (8 * B + 16)) & 0xffu);
    return __builtin_amdgcn_perm(__float_as_uint(b), __float_as_uint(a), 0x07060302u);
  }

  // operand of octet J that takes base and 2^(b-1) off: the same for all lanes
  template <int J>
  __device__ __forceinline__ static void centre(Frag& f) {
#pragma unroll
    for (int i = 0; i < 4; i++) f.u[i] = centre_pair(J, i);
  }
};

}  // namespace matgptq
