// Codes as matrix operands without dequantisation: a pair of codes becomes a pair of storage-type numbers (fp16 or bf16);
// scale and zero point are applied to the product of a whole group.
//
// fp16: with the exponent of 2^(10 - p) a mantissa step is 2^-p, so a field that starts at bit p of the half word reads as
// 2^(10 - p) + c  exactly after a mask and an OR, whatever p is, and a packed addition leaves  c - 2^(b-1).
//
// bf16 has no packed addition.  Its 7 mantissa bits hold  2^(7 - p) + c  as long as the field ends at bit 6, and products
// with that are corrected afterwards by  -(base + 2^(b-1))  times the sum of the activations.  What is taken off again has to
// stay of the size of the codes: where one activation is thousands of times the others (a column of outliers), the rounding
// errors of base times that activation remain in the rows whose weight there is nothing.  So fields are shifted up as far as
// they go: base 16 at 4 bits, 8 at 3, 4 at 2.  Six bits stay at 128 (twice their range), bytes are converted (base 0).
//
// Rows whose weight is zero in a column of activations 10000 times the rest (4096 columns, M = 16, 2 to 8 bits), off by, of the
// size of an output: fp16 2.1e-4 (2.1e-4 to 2.9e-4 with rounded weights; 4.9e-4 to 4.0e-3 with base + code and one base per
// position taken off afterwards), at 60000 times the same; bf16 1.7e-3 (1.7e-3 to 2.3e-3), at 60000 times 1.7e-3 to 2.6e-3.
#pragma once
#include "tile_format.h"

namespace matgptq {

// two equal 16-bit numbers 2^e of the storage type
constexpr uint32_t pow2_pair(int e) {
  const uint32_t h = kBf16 ? (uint32_t)(127 + e) << 7 : (uint32_t)(15 + e) << 10;
  return h | (h << 16);
}
// the negative of the small integer v > 0 (exact in either storage type), twice
constexpr uint32_t minus_pair(int v) {
  int e = 0;
  while ((v >> (e + 1)) != 0) e++;
  const uint32_t h = kBf16 ? ((uint32_t)(127 + e) << 7) | ((uint32_t)(v << (7 - (e < 7 ? e : 7))) & 0x7fu)
                           : ((uint32_t)(15 + e) << 10) | ((uint32_t)(v << (10 - e)) & 0x3ffu);
  return (h | 0x8000u) * 0x10001u;
}

template <int BITS, bool MASTER>
struct RawOperand {
  using Fmt = TileFormat<BITS, MASTER>;
  static constexpr bool kNibbles = BITS == 3 || BITS == 4 || (MASTER && BITS == 2);
  static constexpr bool kCentred = !kBf16;  // operands are c - 2^(b-1); else base + c, the same base for all of them
  static constexpr int kMant = kBf16 ? 7 : 10;
  // Bit of the half word that the field of pair i is masked at, octet j.
  static constexpr int pos(int j, int i) {
    if (BITS == 8 || (MASTER && BITS == 6)) return 0;
    if (kBf16) return BITS == 6 ? 0 : BITS == 4 ? 3 : kNibbles ? 4 : 5;
    if (BITS != 2 || MASTER) return (i & 1) ? 4 : 0;
    return (j & 1) == 0 ? 2 * i : i == 0 ? 8 : 2 * i + 2;  // 2 bits: field f at bit 2f, from field 5 on six bits down
  }
  static constexpr int kBase = kCentred || BITS == 8 ? 0 : 1 << (kMant - pos(0, 0));
  static constexpr uint32_t kOff = minus_pair(kBase + (1 << (BITS - 1)));  // !kCentred: operand that takes base and 2^(b-1) off

  static constexpr int kSteps = kBf16 || BITS == 8 || (MASTER && BITS == 6) ? 1 : BITS == 2 && !MASTER ? 5 : 2;  // positions in use
  static constexpr int kWidth = BITS == 2 && !MASTER ? 2 : 4;  // bits between them
  uint32_t g[kSteps];  // VGPRs: pairs of 2^(kMant - p)
  uint32_t m[kSteps];  // SGPRs: masks of a pair of fields
  uint32_t s[kSteps];  // SGPRs: pairs of -(2^(kMant - p) + 2^(b-1))
  uint32_t t[2];       // SGPRs: masks of the third bits (3 bits), of the upper four bits (6 bits)
  __device__ __forceinline__ RawOperand() {
    for (int i = 0; i < kSteps; i++) {
      const int p = kSteps == 1 ? pos(0, 0) : i * kWidth;
      g[i] = opaque_vgpr(pow2_pair(kMant - p));
      m[i] = opaque_sgpr((kNibbles ? BITS == 4 ? 0x000F000Fu : 0x00070007u : 0x00030003u) << p);
      s[i] = kCentred ? opaque_sgpr(minus_pair((1 << (kMant - p)) + (1 << (BITS - 1)))) : 0u;
    }
    t[0] = opaque_sgpr(BITS == 3 ? 0x44444444u : 0x003C003Cu);
    t[1] = opaque_sgpr(0x03C003C0u);
  }

  static constexpr int step(int p) { return kSteps == 1 ? 0 : p / kWidth; }
  // x moved from bit FROM of the half words to bit TO (what is not masked away afterwards)
  template <int FROM, int TO>
  __device__ __forceinline__ static uint32_t moved(uint32_t x) {
    return FROM > TO ? x >> (FROM - TO) : FROM < TO ? x << (TO - FROM) : x;
  }
  // the field at bit P, as 2^(kMant - P) + field
  template <int P>
  __device__ __forceinline__ uint32_t field(uint32_t x) const {
    return and_or(x, m[step(P)], g[step(P)]);
  }
  template <int P>
  __device__ __forceinline__ uint32_t centred(uint32_t pair) const {
    if constexpr (!kCentred) return pair;
    return __builtin_bit_cast(uint32_t, h2_from_bits(pair) + h2_from_bits(s[step(P)]));
  }

  // the four pairs of octet J
  template <int J>
  __device__ __forceinline__ void octet(const uint32_t (&w)[Fmt::kWords], uint32_t (&r)[4]) const {
    constexpr int p0 = pos(J, 0), p1 = pos(J, 1), p2 = pos(J, 2), p3 = pos(J, 3);
    if constexpr (kNibbles) {
      uint32_t x;
      if constexpr (MASTER) {
        x = master_nibble_word<BITS, J>(w);
      } else if constexpr (BITS == 4) {
        x = w[J];
      } else {
        const uint32_t low = (w[J >> 1] >> (2 * (J & 1))) & 0x33333333u;
        const uint32_t c = w[2];
        x = and_or(J == 0 ? (c << 2) : J == 1 ? (c << 1) : J == 2 ? c : (c >> 1), t[0], low);
      }
      r[0] = field<p0>(moved<0, p0>(x));
      r[1] = field<p1>(moved<4, p1>(x));
      r[2] = field<p2>(moved<8, p2>(x));
      r[3] = field<p3>(moved<12, p3>(x));
    } else if constexpr (BITS == 2) {
      // sixteen fields of two bits, field f of each half word at bit 2f; octet 2d holds fields 0..3, octet 2d + 1 fields 4..7
      const uint32_t x = w[J >> 1];
      constexpr int first = 8 * (J & 1);
      r[0] = field<p0>(moved<first, p0>(x));
      r[1] = field<p1>(moved<first + 2, p1>(x));
      r[2] = field<p2>(moved<first + 4, p2>(x));
      r[3] = field<p3>(moved<first + 6, p3>(x));
    } else if constexpr (BITS == 6 && !MASTER) {
      // the upper four bits of pair i at bit 4i, two lower than in the code; the lower two at bits 0, 4, 2, 6
      const uint32_t h = w[J], l = (J & 1) ? (w[4 + (J >> 1)] >> 8) : w[4 + (J >> 1)];
      constexpr int up1 = p1 ? 1 : 0;
      // (the inner result is hidden from the optimiser, which would regroup the two instructions)
      r[0] = and_or(moved<0, p0 + 2>(h), t[0], opaque_vgpr(field<p0>(moved<0, p0>(l))));
      r[1] = and_or(moved<4, p1 + 2>(h), t[up1], opaque_vgpr(field<p1>(moved<4, p1>(l))));
      r[2] = and_or(moved<8, p2 + 2>(h), t[0], opaque_vgpr(field<p2>(moved<2, p2>(l))));
      r[3] = and_or(moved<12, p3 + 2>(h), t[up1], opaque_vgpr(field<p3>(moved<6, p3>(l))));
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
      constexpr int b1 = MASTER ? 0 : 1, b2 = MASTER ? 1 : 0;
      r[0] = bytes<0>(a);
      r[1] = bytes<b1>(MASTER ? b : a);
      r[2] = bytes<b2>(MASTER ? a : b);
      r[3] = bytes<1>(b);
    }
    r[0] = centred<p0>(r[0]);
    r[1] = centred<p1>(r[1]);
    r[2] = centred<p2>(r[2]);
    r[3] = centred<p3>(r[3]);
  }

  // bytes B and B + 2 of x, as base + byte
  template <int B>
  __device__ __forceinline__ static uint32_t bytes(uint32_t x) {
    if constexpr (kBf16 && BITS == 8) {  // eight significant bits: the upper half of the fp32 number is exact
      const float a = (float)((x >> (8 * B)) & 0xffu), b = (float)((x >> (8 * B + 16)) & 0xffu);
      return __builtin_amdgcn_perm(__float_as_uint(b), __float_as_uint(a), 0x07060302u);
    }
    return __builtin_amdgcn_perm(kBf16 ? 0x43434343u : 0x64646464u, x, B ? 0x04030401u : 0x04020400u);
  }
};

}  // namespace matgptq
