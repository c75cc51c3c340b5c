// Few-rows kernel: one to sixteen batch rows, one scale per tile of 128 columns or per row.
// Compiled once per bitwidth with -DMATGPTQ_BITS=b.
// Role of the reference's small-batch kernels (inference_lib/matgptq_cuda/csrc/matgptq_gemm.cu:337-953).
//
//  * Eight waves own R row blocks of 16 weight rows and all of K; wave w walks the K tiles w, w + 8, ...  The activations of a
//    tile are copied with buffer_load ... lds into the wave's own buffer (256 contiguous bytes per 16 lanes, 16-byte chunk c
//    of row r at position c ^ r), codes, scales and zeros go to registers.  Two buffers and two register sets: tile t + 2 is
//    requested while t is multiplied and t + 1 is on its way.  Walks of one tile (K up to 1024) have one of each, half the
//    registers, and more workgroups per CU.  Buffers hold 4, 8 or 16 batch rows.
//  * Codes are matrix operands as they are (raw_operand.h): a mask and an OR per pair of codes, no weight is formed.  The
//    activations are the 16-row operand, the 16 weight rows the columns, so lane (n, q) ends with batch rows 4q .. 4q+3 of
//    weight row n and applies that row's one scale to the four sums.  What the operand carries besides the code, and the zero
//    point, multiply sums of activations only: two chains of four MFMAs against constants per tile, shared by the R row
//    blocks, whose result is the start value of the code chain.  Per tile and row block that leaves some 30 vector
//    instructions at 4 bits (the mid-batch kernel, which forms weights, has 50, on bf16 storage 66), and no rounded weight:
//    the error against 64 bits is that of the result's rounding (fp16 2.1e-4, 2.8e-4 with rounded weights; bf16 1.7e-3, 2.2e-3).
//  * What bounds it: the copies of the activations, which every workgroup repeats, and HBM.  On layers with one row block per
//    CU and a long K the copies are most of the traffic of a CU (4096 x 14336 at M = 16: 458 KB beside 115 KB of codes).
//
// Measured against what ran before, weights cold, us (mid-batch kernel; * gemv kernel, which stages activations through
// registers once per wave and row block):
//   28672 x 4096  3 bits bf16  M = 8  17.9 -> 12.7    4 bits fp16  M = 8  16.1 -> 14.2,  M = 16  16.9 -> 15.5
//    4096 x 14336 3 bits bf16  M = 8  11.1* -> 9.4    4 bits fp16  M = 16 13.2 -> 12.9
//    4096 x 4096  3 bits bf16  M = 8   5.4* -> 4.5    4 bits fp16  M = 16  5.8 -> 5.4
//    8192 x 3584  4 bits fp16  M = 16  7.2 -> 6.7     1280 x 8192  4 bits fp16  M = 16  7.8 -> 7.0
// and over 10000 random calls (every bitwidth and storage type, K = 256 .. 16384, M = 5 .. 16) 1.08 to 1.45 times faster on
// the geometric mean of each format, slower by more than 1.5 % on one in a thousand.
// Tried and taken back: activations loaded straight into the operand (16 rows x 64 bytes per load: 4096 x 14336 at M = 16
// 13 -> 17 us), four buffers and everything requested at the start (28672 x 4096: within 3 % either way), sixteen waves
// (ahead only below 5 rows on walks past 8192 columns), consecutive tiles per wave (2 % slower).
#include "fewrows_plan.h"
#include "raw_operand.h"

#ifndef MATGPTQ_BITS
#error "compile with -DMATGPTQ_BITS={2,3,4,6,8}"
#endif

namespace matgptq {

namespace {

constexpr int kBits = MATGPTQ_BITS;
constexpr int kWaves = kFewRowsWaves;

// Waves per SIMD to hold the registers to: four while the sets of codes, scales and zeros and the sums leave room for what
// one tile needs (some 60).
constexpr int few_rows_min_waves(int bits, bool zp, int r, bool master, bool one) {
  const int words = master ? master_words(bits) : bits;
  return (one ? 1 : 2) * r * (words + 1 + (zp ? 1 : 0)) + 4 * r <= 64 ? 4 : 2;
}

// ROWS: batch rows held per tile, 8 or 16 (rows beyond M are never stored, whatever they hold)
// ONE: walks of one tile, which need one buffer and one register set
template <int BITS, int GROUP, bool ZP, int R, int ROWS, bool MASTER, bool ONE>
__global__ void __launch_bounds__(64 * kWaves, few_rows_min_waves(BITS, ZP, R, MASTER, ONE))
few_rows_kernel(const GemmArgs a) {
  static_assert(GROUP == 128 || GROUP == -1, "one scale per tile or row");
  using Fmt = TileFormat<BITS, MASTER>;
  using Raw = RawOperand<BITS, MASTER>;
  constexpr int kStage = ROWS * 256;  // bytes of one activation buffer of a wave
  constexpr int kCopies = ROWS / 4;
  constexpr int kSums = kWaves * R * 1024;  // the waves' sums reuse the first buffers
  constexpr float kMul = (float)(1 << (8 - BITS));
  __shared__ __align__(16) unsigned char smem_even[kWaves * kStage > kSums ? kWaves * kStage : kSums];
  // (an array of its own: the compiler orders LDS copies and reads per variable)
  __shared__ __align__(16) unsigned char smem_odd[ONE ? 16 : kWaves * kStage];

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r16 = lane & 15;
  const int q = lane >> 4;
  const int rb_first = blockIdx.x * R;

  constexpr uint32_t tile_bytes = Fmt::kTileBytes;
  const uint32_t rb_bytes = (uint32_t)a.k_tiles * tile_bytes;
  const uint32_t w_bytes = (uint32_t)a.row_blocks * rb_bytes;
  const uint32_t aux_bytes = (uint32_t)a.row_blocks * a.G * 32;  // scales / zeros: [N/16][G][16] halves
  const uint32_t x_bytes = (uint32_t)a.M * (uint32_t)a.K * 2u;

  float4v acc[R];
#pragma unroll
  for (int rr = 0; rr < R; rr++) acc[rr] = float4v{0.f, 0.f, 0.f, 0.f};
  float4v xsum = {0.f, 0.f, 0.f, 0.f};  // one scale per row with zero points: sums of all activations

  const Raw raw;
  Frag centre[Raw::kOddOctets ? 2 : 1], ones;
  Raw::template centre<0>(centre[0]);
  if constexpr (Raw::kOddOctets) Raw::template centre<1>(centre[1]);
#pragma unroll
  for (int i = 0; i < 4; i++) ones.u[i] = pow2_pair(0);
  auto mma = [](const Frag& x, const Frag& w, float4v c) {
    if constexpr (kBf16)
      return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, x.h), __builtin_bit_cast(bf16x8, w.h), c, 0, 0, 0);
    else
      return __builtin_amdgcn_mfma_f32_16x16x32_f16(x.h, w.h, c, 0, 0, 0);
  };

  // codes, scales and zeros of the tile in use and of the next one (scales and zeros as loaded)
  uint32_t wr[ONE ? 1 : 2][R][Fmt::kWords], sr[ONE ? 1 : 2][R], zr[ONE ? 1 : 2][R];
  auto load_weights = [&](uint32_t (&w)[R][Fmt::kWords], uint32_t (&s)[R], uint32_t (&z)[R], int kb) {
#pragma unroll
    for (int rr = 0; rr < R; rr++) {
      const int rb = rb_first + rr;
      const bool valid = rb < a.row_blocks && kb < a.k_tiles;
      const BufRsrc wr = make_rsrc(a.packed, valid ? w_bytes : 0u);
      Fmt::load(wr, (uint32_t)rb * rb_bytes + (uint32_t)kb * tile_bytes, lane, w[rr]);
      if constexpr (GROUP != -1) {
        const BufRsrc sr = make_rsrc(a.scales, valid ? aux_bytes : 0u);
        const uint32_t so = ((uint32_t)rb * a.G + (uint32_t)kb) * 32;  // bytes
        s[rr] = __builtin_amdgcn_raw_buffer_load_b16(sr, r16 * 2, so, 0);
        if constexpr (ZP) {
          const BufRsrc zr = make_rsrc(a.zeros, valid ? aux_bytes : 0u);
          z[rr] = __builtin_amdgcn_raw_buffer_load_b16(zr, r16 * 2, so, 0);
        }
      }
    }
    __builtin_amdgcn_sched_barrier(0);
  };

  // Copy of one tile's activations: instruction i moves rows 4i .. 4i+3 (lane l: row 4i + l/16, LDS position
  // l%16, which holds chunk (l%16) ^ row of the row's 256 bytes).
  uint32_t copy_off[kCopies];
#pragma unroll
  for (int i = 0; i < kCopies; i++) {
    const int row = 4 * i + q;
    copy_off[i] = row < a.M ? (uint32_t)row * (uint32_t)a.K * 2u + (r16 ^ row) * 16 : x_bytes;
  }
  auto copy_x = [&](unsigned char* to, int kb) {
    const BufRsrc xres = make_rsrc(a.x, kb < a.k_tiles ? x_bytes : 0u);
#pragma unroll
    for (int i = 0; i < kCopies; i++)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(xres, (__attribute__((address_space(3))) void*)(to + i * 1024), 16, (int)copy_off[i],
                                               (int)((uint32_t)kb * 256u), 0, 0);
    __builtin_amdgcn_sched_barrier(0);
  };

  unsigned char* const stage_even = smem_even + wave * kStage;
  unsigned char* const stage_odd = smem_odd + (ONE ? 0 : wave * kStage);
  const int xrow = r16 & (ROWS - 1);
  constexpr int kLoads = kCopies + R * ((MASTER ? master_load_count(BITS) : tile_load_count(BITS)) + (GROUP == -1 ? 0 : ZP ? 2 : 1));
  static_assert(kLoads < 64, "vmcnt counts up to 63");
  // Tile t of the walk (K tile wave + 8 t) in buffer and register set `btag`.  `moretag`: tile t + 2 is requested;
  // without it (the last two tiles) set 0 leaves set 1's requests in flight, set 1 none.
  auto tile = [&](int t, auto btag, auto moretag) {
    constexpr int B = decltype(btag)::value;
    constexpr bool kMore = decltype(moretag)::value;
    constexpr int kYounger = !ONE && (kMore || B == 0) ? kLoads : 0;  // requests of the tile behind this one
    const int kb = wave + t * kWaves;
    unsigned char* const buf = B == 0 ? stage_even : stage_odd;
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_waitcnt((kYounger & 15) | (7 << 4) | (15 << 8) | ((kYounger >> 4) << 14));
    __builtin_amdgcn_sched_barrier(0);
    Frag xf[4];
#pragma unroll
    for (int j = 0; j < 4; j++) xf[j].v = *reinterpret_cast<const uint4*>(buf + xrow * 256 + (((4 * j + q) ^ xrow) * 16));
    __builtin_amdgcn_sched_barrier(0);
    if constexpr (kMore) {
      __builtin_amdgcn_s_waitcnt(15 | (7 << 4) | (0 << 8) | (3 << 14));  // lgkmcnt(0): the buffer is free
      __builtin_amdgcn_sched_barrier(0);
      copy_x(buf, kb + 2 * kWaves);
    }
    // (only the last tile of a walk can lie beyond K; its buffer may hold anything)
    if (kMore || kb < a.k_tiles) {
      const float4v zero4 = {0.f, 0.f, 0.f, 0.f};
      float4v off = zero4, xs = zero4;
#pragma unroll
      for (int j = 0; j < 4; j++) {
        off = mma(xf[j], centre[Raw::kOddOctets ? (j & 1) : 0], off);
        if constexpr (ZP) xs = mma(xf[j], ones, xs);
      }
      if constexpr (ZP && GROUP == -1) xsum += xs;
#pragma unroll
      for (int rr = 0; rr < R; rr++) {
        float4v d = off;
        if constexpr (GROUP == -1) {
          d += acc[rr];
        } else if constexpr (ZP) {
          const float z = 128.0f / kMul - storage_to_float((uint16_t)zr[B][rr]) * (1.0f / kMul);
#pragma unroll
          for (int e = 0; e < 4; e++) d[e] = __builtin_fmaf(z, xs[e], d[e]);
        }
        auto one = [&](auto jtag) {
          constexpr int J = decltype(jtag)::value;
          Frag codes;
          raw.template octet<J>(wr[B][rr], codes.u);
          d = mma(xf[J], codes, d);
        };
        one(std::integral_constant<int, 0>{});
        one(std::integral_constant<int, 1>{});
        one(std::integral_constant<int, 2>{});
        one(std::integral_constant<int, 3>{});
        if constexpr (GROUP == -1) {
          acc[rr] = d;
        } else {
          const float s = storage_to_float((uint16_t)sr[B][rr]);
#pragma unroll
          for (int e = 0; e < 4; e++) acc[rr][e] = __builtin_fmaf(s, d[e], acc[rr][e]);
        }
      }
    }
    __builtin_amdgcn_sched_barrier(0);
    if constexpr (kMore) load_weights(wr[B], sr[B], zr[B], kb + 2 * kWaves);
  };

  const int walk = (a.k_tiles + kWaves - 1) / kWaves;  // tiles of the longest walk
  using Even = std::integral_constant<int, 0>;
  using Odd = std::integral_constant<int, 1>;
  __builtin_amdgcn_sched_barrier(0);
  copy_x(stage_even, wave);
  load_weights(wr[0], sr[0], zr[0], wave);
  if constexpr (ONE) {
    tile(0, Even{}, std::false_type{});
  } else {
    copy_x(stage_odd, wave + kWaves);
    load_weights(wr[1], sr[1], zr[1], wave + kWaves);
    int t = 0;
    for (; t + 2 < walk; t += 2) {
      tile(t, Even{}, std::true_type{});
      tile(t + 1, Odd{}, std::true_type{});
    }
    tile(t, Even{}, std::false_type{});
    if (t + 1 < walk) tile(t + 1, Odd{}, std::false_type{});
  }

  // Infinities and NaN among the activations (and bf16 numbers beyond 2^120) have met `base` times themselves with the
  // other sign and left NaN: such a wave forms its sums again, with dequantised weights as the other kernels do.
  bool finite = true;
#pragma unroll
  for (int rr = 0; rr < R; rr++)
#pragma unroll
    for (int e = 0; e < 4; e++) finite = finite && __builtin_isfinite(acc[rr][e]);
  const bool again = __builtin_amdgcn_ballot_w64(!finite) != 0;
  if (again) {
    const typename Fmt::Consts unpack;
    const uint32_t x_off = xrow < a.M ? (uint32_t)xrow * (uint32_t)a.K * 2u + q * 16 : x_bytes;
    const BufRsrc xres = make_rsrc(a.x, x_bytes);
#pragma unroll
    for (int rr = 0; rr < R; rr++) acc[rr] = float4v{0.f, 0.f, 0.f, 0.f};
    for (int kb = wave; kb < a.k_tiles; kb += kWaves) {
#pragma unroll
      for (int rr = 0; rr < R; rr++) {
        const int rb = rb_first + rr < a.row_blocks ? rb_first + rr : a.row_blocks - 1;
        uint32_t w[Fmt::kWords];
        Fmt::load(make_rsrc(a.packed, w_bytes), (uint32_t)rb * rb_bytes + (uint32_t)kb * tile_bytes, lane, w);
        const size_t g = ((size_t)rb * a.G + (GROUP == -1 ? 0 : kb)) * 16 + r16;
        const float s = storage_to_float(a.scales[g]);
        const float z = ZP ? s * (storage_to_float(a.zeros[g]) - 128.0f) : __uint_as_float(opaque_vgpr(0u));
        auto one = [&](auto jtag) {
          constexpr int J = decltype(jtag)::value;
          const u32x4 v = __builtin_amdgcn_raw_buffer_load_b128(xres, x_off, (uint32_t)kb * 256u + J * 64u, 0);
          Frag x, aw;
          x.v = make_uint4(v.x, v.y, v.z, v.w);
          if constexpr (kBf16) {
            dequant_octet_bf16_fmt<Fmt, BITS, J>(w, unpack, s * kMul, z, aw);
          } else {
            const _Float16 s1 = (_Float16)(s * kMul), z1 = (_Float16)z;
            dequant_octet_fmt<Fmt, BITS, J, true>(w, unpack, half2v{z1, z1}, half2v{s1, s1}, aw);
          }
          acc[rr] = mma(x, aw, acc[rr]);
        };
        one(std::integral_constant<int, 0>{});
        one(std::integral_constant<int, 1>{});
        one(std::integral_constant<int, 2>{});
        one(std::integral_constant<int, 3>{});
      }
    }
#pragma unroll
    for (int rr = 0; rr < R; rr++) acc[rr] *= 1.0f / kMul;
  }

  if (GROUP == -1 && !again) {  // the row's one scale and zero point
#pragma unroll
    for (int rr = 0; rr < R; rr++) {
      const int rb = rb_first + rr < a.row_blocks ? rb_first + rr : a.row_blocks - 1;
      const float s = storage_to_float(a.scales[(size_t)rb * 16 + r16]);
      if constexpr (ZP) {
        const float z = 128.0f / kMul - storage_to_float(a.zeros[(size_t)rb * 16 + r16]) * (1.0f / kMul);
#pragma unroll
        for (int e = 0; e < 4; e++) acc[rr][e] = __builtin_fmaf(z, xsum[e], acc[rr][e]);
      }
      // (a sum times scale 0 is +0, as a sum of products with it is)
#pragma unroll
      for (int e = 0; e < 4; e++) acc[rr][e] = __builtin_fmaf(s, acc[rr][e], 0.f);
    }
  }

  // The waves' sums of every output meet in LDS (over the activation buffers: every wave has to be done with its
  // own first), four batch rows 4q .. 4q+3 of weight row r16 per lane and row block.
  __builtin_amdgcn_s_waitcnt(0 | (7 << 4) | (0 << 8) | (0 << 14));  // nothing in flight into LDS any more
  __syncthreads();
  float* const red = reinterpret_cast<float*>(smem_even);
#pragma unroll
  for (int rr = 0; rr < R; rr++) *reinterpret_cast<float4v*>(red + ((wave * R + rr) * 64 + lane) * 4) = acc[rr];
  __syncthreads();
  for (int o = tid; o < R * 256; o += 64 * kWaves) {
    float sum = red[o];
#pragma unroll
    for (int w = 1; w < kWaves; w++) sum += red[w * R * 256 + o];
    const int l = (o >> 2) & 63;
    const int rb = rb_first + (o >> 8), m = 4 * (l >> 4) + (o & 3);
    if (rb < a.row_blocks && m < a.M) a.y[(size_t)m * a.N + (size_t)rb * 16 + (l & 15)] = float_to_storage(sum * kMul);
  }
}

template <int GROUP, bool ZP, int R, int ROWS, bool MASTER>
hipError_t launch_r(const GemmArgs& a, hipStream_t stream) {
  const dim3 grid((a.row_blocks + R - 1) / R), block(64 * kWaves);
  if (a.k_tiles <= kWaves)
    hipLaunchKernelGGL((few_rows_kernel<kBits, GROUP, ZP, R, ROWS, MASTER, true>), grid, block, 0, stream, a);
  else
    hipLaunchKernelGGL((few_rows_kernel<kBits, GROUP, ZP, R, ROWS, MASTER, false>), grid, block, 0, stream, a);
  return hipGetLastError();
}

template <int GROUP, bool ZP, int R, bool MASTER>
hipError_t launch_batch(const GemmArgs& a, hipStream_t stream) {
  if (a.M <= 4) return launch_r<GROUP, ZP, R, 4, MASTER>(a, stream);
  return a.M <= 8 ? launch_r<GROUP, ZP, R, 8, MASTER>(a, stream) : launch_r<GROUP, ZP, R, 16, MASTER>(a, stream);
}

template <int GROUP, bool ZP, bool MASTER>
hipError_t launch_rows(const GemmArgs& a, int r, hipStream_t s) {
  // (four row blocks of 8-bit codes, or of six and eight planes, do not fit the registers)
  if constexpr (kBits <= (MASTER ? 4 : 6)) {
    if (r >= 4) return launch_batch<GROUP, ZP, 4, MASTER>(a, s);
  }
  if (r >= 2) return launch_batch<GROUP, ZP, 2, MASTER>(a, s);
  return launch_batch<GROUP, ZP, 1, MASTER>(a, s);
}

template <int GROUP, bool ZP>
hipError_t launch_storage(const GemmArgs& a, int r, bool master, hipStream_t s) {
  return master ? launch_rows<GROUP, ZP, true>(a, r, s) : launch_rows<GROUP, ZP, false>(a, r, s);
}

}  // namespace

#define MATGPTQ_CAT2(a, b) a##b
#define MATGPTQ_CAT(a, b) MATGPTQ_CAT2(a, b)
#if MATGPTQ_BF16
#define MATGPTQ_LAUNCH_NAME MATGPTQ_CAT(MATGPTQ_CAT(launch_few_rows_b, MATGPTQ_BITS), _bf16)
#else
#define MATGPTQ_LAUNCH_NAME MATGPTQ_CAT(launch_few_rows_b, MATGPTQ_BITS)
#endif
// M <= 16, group size 128 or -1.  r: row blocks of 16 weight rows per workgroup (1, 2 or 4); master: `a.packed` holds
// master-resident bit planes
hipError_t MATGPTQ_LAUNCH_NAME(const GemmArgs& a, int group_size, int r, bool master, hipStream_t stream) {
  const bool zp = a.zeros != nullptr;
  if (a.M > 16 || group_size == 32) return hipErrorInvalidValue;
  if (group_size == 128)
    return zp ? launch_storage<128, true>(a, r, master, stream) : launch_storage<128, false>(a, r, master, stream);
  return zp ? launch_storage<-1, true>(a, r, master, stream) : launch_storage<-1, false>(a, r, master, stream);
}

}  // namespace matgptq
