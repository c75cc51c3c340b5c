// Slicing and packing of a lane slot's 32 codes four at a time, on the bytes of 32-bit words (the
// load-time kernels).  Same results as slice_code / Codec<b>::encode_lane / master_encode_lane of
// layout.h and master_layout.h, which the host packer runs one code after another.
//
// A slot arrives as four octets of eight bytes (element e of an octet = byte e).  Two byte permutes
// bring an octet into the order of the packed fields:
//     A = (e0, e4, e1, e5),  B = (e2, e6, e3, e7)   (byte 0 first)
// so that A | B << 4 of values below 16 is the nibble word of layout.h (element e in nibble
// nibble_of(e)), and A, B are the byte words h = 0, 1 of master_layout.h.
#pragma once
#include "device_common.h"
#include "master_layout.h"

namespace matgptq {

struct OctetBytes {
  uint32_t a, b;
};

__device__ __forceinline__ OctetBytes octet_bytes(uint2 v) {
  return {__builtin_amdgcn_perm(v.y, v.x, 0x05010400u), __builtin_amdgcn_perm(v.y, v.x, 0x07030602u)};
}

// slice_code on the four bytes of a word
template <int BITS>
__device__ __forceinline__ uint32_t slice_bytes(uint32_t v) {
  if constexpr (BITS == 8) return v;
  constexpr uint32_t k1 = 0x01010101u, top = k1 * ((1u << BITS) - 1u);
  const uint32_t s = ((v >> (8 - BITS)) & top) + ((v >> (7 - BITS)) & k1);  // 0 .. 2^b per byte
  return s - ((s >> BITS) & k1);                                            // 2^b -> 2^b - 1
}

// Codes already sliced: what lies above the low b bits is dropped, as encode_lane drops it.
template <int BITS>
__device__ __forceinline__ uint32_t low_bytes(uint32_t v) {
  if constexpr (BITS == 8) return v;
  return v & (0x01010101u * ((1u << BITS) - 1u));
}

// nibble words of the four octets -> the packed words (2, 3 and 4 bits)
template <int BITS>
__device__ __forceinline__ void pack_nibble_words(const uint32_t (&x)[4], uint32_t (&w)[BITS]) {
  static_assert(BITS <= 4, "nibble form");
  if constexpr (BITS == 4) {
#pragma unroll
    for (int j = 0; j < 4; j++) w[j] = x[j];
  } else if constexpr (BITS == 3) {
    w[0] = (x[0] & 0x33333333u) | ((x[1] & 0x33333333u) << 2);
    w[1] = (x[2] & 0x33333333u) | ((x[3] & 0x33333333u) << 2);
    w[2] = ((x[0] >> 2) & 0x11111111u) | ((x[1] >> 1) & 0x22222222u) | (x[2] & 0x44444444u) |
           ((x[3] << 1) & 0x88888888u);
  } else {
    uint32_t z[4];  // even elements' fields in the low byte of the low half, odd ones' in that of the high half
#pragma unroll
    for (int j = 0; j < 4; j++) {
      const uint32_t y = (x[j] | (x[j] >> 2)) & 0x0F0F0F0Fu;
      z[j] = (y | (y >> 4)) & 0x00FF00FFu;
    }
    w[0] = z[0] | (z[1] << 8);
    w[1] = z[2] | (z[3] << 8);
  }
}

// byte words of the four octets -> the packed words (6 and 8 bits)
template <int BITS>
__device__ __forceinline__ void pack_byte_words(const OctetBytes (&o)[4], uint32_t (&w)[BITS]) {
  static_assert(BITS == 6 || BITS == 8, "byte form");
  if constexpr (BITS == 8) {
#pragma unroll
    for (int j = 0; j < 4; j++) {
      w[2 * j] = __builtin_amdgcn_perm(o[j].b, o[j].a, 0x06020400u);      // e0 e2 e1 e3
      w[2 * j + 1] = __builtin_amdgcn_perm(o[j].b, o[j].a, 0x07030501u);  // e4 e6 e5 e7
    }
  } else {
    uint32_t z[4];
#pragma unroll
    for (int j = 0; j < 4; j++) {
      w[j] = ((o[j].a >> 2) & 0x0F0F0F0Fu) | ((o[j].b << 2) & 0xF0F0F0F0u);
      const uint32_t y = (o[j].a & 0x03030303u) | ((o[j].b & 0x03030303u) << 4);
      z[j] = (y | (y >> 6)) & 0x00FF00FFu;
    }
    w[4] = z[0] | (z[1] << 8);
    w[5] = z[2] | (z[3] << 8);
  }
}

// four octets of bytes -> the packed words; SLICE: the bytes are 8-bit master codes
template <int BITS, bool SLICE>
__device__ __forceinline__ void pack_slot(const uint2 (&v)[4], uint32_t (&w)[BITS]) {
  OctetBytes o[4];
#pragma unroll
  for (int j = 0; j < 4; j++) {
    o[j] = octet_bytes(v[j]);
    o[j].a = SLICE ? slice_bytes<BITS>(o[j].a) : low_bytes<BITS>(o[j].a);
    o[j].b = SLICE ? slice_bytes<BITS>(o[j].b) : low_bytes<BITS>(o[j].b);
  }
  if constexpr (BITS <= 4) {
    uint32_t x[4];
#pragma unroll
    for (int j = 0; j < 4; j++) x[j] = o[j].a | (o[j].b << 4);
    pack_nibble_words<BITS>(x, w);
  } else {
    pack_byte_words<BITS>(o, w);
  }
}

// four octets of master codes -> the eight plane words of master_layout.h
__device__ __forceinline__ void pack_slot_planes(const uint2 (&v)[4], uint32_t (&w)[8]) {
  constexpr uint32_t k1 = 0x11111111u, k3 = 0x33333333u;
  uint32_t hi[4], lo[4];  // nibble words of the upper and the lower four bits
#pragma unroll
  for (int j = 0; j < 4; j++) {
    const OctetBytes o = octet_bytes(v[j]);
    hi[j] = ((o.a >> 4) & 0x0F0F0F0Fu) | (o.b & 0xF0F0F0F0u);
    lo[j] = (o.a & 0x0F0F0F0Fu) | ((o.b << 4) & 0xF0F0F0F0u);
  }
#pragma unroll
  for (int i = 2; i < 6; i++) w[i] = 0;
#pragma unroll
  for (int d = 0; d < 2; d++) {
    w[d] = ((hi[2 * d] >> 2) & k3) | (hi[2 * d + 1] & (k3 << 2));
    w[6 + d] = (lo[2 * d] & k3) | ((lo[2 * d + 1] & k3) << 2);
  }
#pragma unroll
  for (int j = 0; j < 4; j++) {
    w[2] |= ((hi[j] >> 1) & k1) << j;
    w[3] |= (hi[j] & k1) << j;
    w[4] |= ((lo[j] >> 3) & k1) << j;
    w[5] |= ((lo[j] >> 2) & k1) << j;
  }
}

// plane words -> the packed words of the b-bit slice
template <int BITS>
__device__ __forceinline__ void pack_slot_from_planes(const uint32_t (&p)[8], uint32_t (&w)[BITS]) {
  if constexpr (BITS <= 4) {
    const uint32_t x[4] = {master_nibble_word<BITS, 0>(p), master_nibble_word<BITS, 1>(p), master_nibble_word<BITS, 2>(p),
                           master_nibble_word<BITS, 3>(p)};
    pack_nibble_words<BITS>(x, w);
  } else {
    const OctetBytes o[4] = {{master_byte_word<BITS, 0, 0>(p), master_byte_word<BITS, 0, 1>(p)},
                             {master_byte_word<BITS, 1, 0>(p), master_byte_word<BITS, 1, 1>(p)},
                             {master_byte_word<BITS, 2, 0>(p), master_byte_word<BITS, 2, 1>(p)},
                             {master_byte_word<BITS, 3, 0>(p), master_byte_word<BITS, 3, 1>(p)}};
    pack_byte_words<BITS>(o, w);
  }
}

// the words of one lane slot to its tile, one store per segment
template <int BITS>
__device__ __forceinline__ void store_tile_words(uint32_t* __restrict__ tile, int lane, const uint32_t (&w)[BITS]) {
  if constexpr (BITS == 2) {
    *reinterpret_cast<uint2*>(tile + lane * 2) = make_uint2(w[0], w[1]);
  } else if constexpr (BITS == 3) {
    *reinterpret_cast<uint2*>(tile + lane * 2) = make_uint2(w[0], w[1]);
    tile[128 + lane] = w[2];
  } else {
    *reinterpret_cast<uint4*>(tile + lane * 4) = make_uint4(w[0], w[1], w[2], w[3]);
    if constexpr (BITS == 6) *reinterpret_cast<uint2*>(tile + 256 + lane * 2) = make_uint2(w[4], w[5]);
    if constexpr (BITS == 8) *reinterpret_cast<uint4*>(tile + 256 + lane * 4) = make_uint4(w[4], w[5], w[6], w[7]);
  }
}

}  // namespace matgptq
