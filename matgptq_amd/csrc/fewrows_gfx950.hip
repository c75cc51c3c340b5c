// Few-rows kernel: one to 64 batch rows, one scale per tile of 128 columns or per row.
// Compiled once per bitwidth with -DMATGPTQ_BITS=b.
// Role of the reference's small-batch kernels (inference_lib/matgptq_cuda/csrc/matgptq_gemm.cu:337-953).
//
//  * Eight waves own R row blocks of 16 weight rows and all of K; wave w walks the K tiles w, w + 8, ...  The activations of a
//    tile are copied with buffer_load ... lds into the wave's own buffer (256 contiguous bytes per 16 lanes, 16-byte chunk c
//    of row r at position c ^ r), codes, scales and zeros go to registers.  Two buffers and two register sets: tile t + 2 is
//    requested while t is multiplied and t + 1 is on its way.  Walks of one tile (K up to 1024) have one of each, half the
//    registers, and more workgroups per CU.  Buffers hold 4, 8, 16 or 32 batch rows; with 32 there is one buffer (64 KB for the
//    eight waves), refilled as soon as its operands are in registers, and two register sets.
//  * Codes are matrix operands as they are (raw_operand.h), no weight is formed: a mask, an OR and on fp16 storage a packed
//    addition per pair of codes.  The activations are the 16-row operand, the 16 weight rows the columns, so lane (n, q) ends
//    with batch rows 4q .. 4q+3 of weight row n and applies that row's one scale to the four sums.  The zero point, and what
//    the operand of bf16 storage carries besides the code, multiply sums of activations only: chains of four MFMAs against
//    constants per tile, shared by the R row blocks, whose result is the start value of the code chain.  No weight is rounded:
//    the error against 64 bits is that of the result's rounding (fp16 2.1e-4, 2.8e-4 with rounded weights; bf16 1.7e-3, 2.2e-3).
//  * What bounds it: no unit alone.  28672 x 4096, 3 bits bf16, M = 8 (13.8 us): HBM 3.4 TB/s, vector issue 0.41, L2 5.6 TB/s;
//    4096 x 14336 (9.7 us): 2.6, 0.29, 8.6.  It is the chain of a wave (copy, operands, products, sums) over the few tiles of
//    its walk, and the copies of the activations, which every workgroup repeats: on layers with one row block per CU and a long K
//    most of the traffic of a CU (4096 x 14336 at M = 16: 458 KB beside 115 KB of codes).
//
// Measured against what ran before, weights from HBM, us (mid-batch kernel; * gemv kernel, which stages activations through
// registers once per wave and row block):
//   28672 x 4096  3 bits bf16  M = 8  20.6 -> 14.9    4 bits fp16  M = 8  19.6 -> 14.8,  M = 16  19.7 -> 15.6
//    4096 x 14336 3 bits bf16  M = 8  11.3* -> 9.4    4 bits fp16  M = 16 14.5 -> 12.7
//    4096 x 4096  3 bits bf16  M = 8   5.6* -> 4.6    4 bits fp16  M = 16  6.0 -> 5.4,   M = 24   7.4 -> 5.9
//    8192 x 3584  4 bits fp16  M = 16  7.7 -> 6.4     1280 x 8192  4 bits fp16  M = 16  8.5 -> 7.7
//    6144 x 4096  4 bits bf16  M = 32  9.4 -> 8.4     1024 x 4096  4 bits bf16  M = 64  7.4 -> 5.1
// The rule in fewrows_plan.h says for which calls and by how much over random ones.
// Tried and taken back: 64 batch rows per workgroup (no faster than two workgroups of 32), activations loaded straight into
// the operand (16 rows x 64 bytes per load: 4096 x 14336 at M = 16 13 -> 17 us), four buffers and everything requested at the
// start (28672 x 4096: within 3 % either way), sixteen waves (ahead only below 5 rows on walks past 8192 columns), consecutive
// tiles per wave (2 % slower).
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

// ROWS: batch rows of a workgroup, 4, 8, 16 or 32 (rows beyond M are never stored, whatever they hold)
// ONE: walks of one tile, which need one buffer and one register set
template <int BITS, int GROUP, bool ZP, int R, int ROWS, bool MASTER, bool ONE>
__global__ void __launch_bounds__(64 * kWaves, ROWS > 16 ? 2 : few_rows_min_waves(BITS, ZP, R, MASTER, ONE))
few_rows_kernel(const GemmArgs a, int n_tiles, int m_tiles) {
  static_assert(GROUP == 128 || GROUP == -1, "one scale per tile or row");
  using Fmt = TileFormat<BITS, MASTER>;
  using Raw = RawOperand<BITS, MASTER>;
  constexpr int MB = ROWS > 16 ? ROWS / 16 : 1;  // blocks of 16 batch rows
  constexpr bool kTwo = !ONE && MB == 1;         // two buffers
  constexpr int kSets = ONE ? 1 : 2;             // register sets
  constexpr int kStage = ROWS * 256;  // bytes of one activation buffer of a wave
  constexpr int kCopies = ROWS / 4;
  constexpr int kSums = kWaves * R * MB * 1024;  // the waves' sums reuse the first buffers
  constexpr float kMul = (float)(1 << (8 - BITS));
  __shared__ __align__(16) unsigned char smem_even[kWaves * kStage > kSums ? kWaves * kStage : kSums];
  // (an array of its own: the compiler orders LDS copies and reads per variable)
  __shared__ __align__(16) unsigned char smem_odd[kTwo ? kWaves * kStage : 16];

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r16 = lane & 15;
  const int q = lane >> 4;
  // Workgroup ids go round-robin over the 8 XCDs: with several blocks of batch rows they are remapped so that the workgroups
  // of one XCD walk those blocks of the same weight rows and share these in its L2 (against ids as they come: two blocks of
  // batch rows 1.05, three 1.08, four 1.12 on the geometric mean of 10000 random calls; a single one the same either way).
  int lid = blockIdx.x;
  if (m_tiles > 1) {
    const int total = n_tiles * m_tiles, xcd = blockIdx.x & 7, rest = total & 7;
    lid = xcd * (total >> 3) + (xcd < rest ? xcd : rest) + (blockIdx.x >> 3);
  }
  const int nt = lid / m_tiles;
  const int m0 = (lid - nt * m_tiles) * ROWS;
  const int rb_first = nt * R;

  constexpr uint32_t tile_bytes = Fmt::kTileBytes;
  const uint32_t rb_bytes = (uint32_t)a.k_tiles * tile_bytes;
  const uint32_t w_bytes = (uint32_t)a.row_blocks * rb_bytes;
  const uint32_t aux_bytes = (uint32_t)a.row_blocks * a.G * 32;  // scales / zeros: [N/16][G][16] halves
  const uint32_t x_bytes = (uint32_t)a.M * (uint32_t)a.K * 2u;

  float4v acc[R][MB], xsum[MB];  // xsum: one scale per row with zero points, sums of all activations
#pragma unroll
  for (int i = 0; i < MB; i++) {
    xsum[i] = float4v{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int rr = 0; rr < R; rr++) acc[rr][i] = float4v{0.f, 0.f, 0.f, 0.f};
  }

  const Raw raw;
  Frag minus, ones;
#pragma unroll
  for (int i = 0; i < 4; i++) {
    minus.u[i] = Raw::kOff;
    ones.u[i] = pow2_pair(0);
  }
  auto mma = [](const Frag& x, const Frag& w, float4v c) {
    if constexpr (kBf16)
      return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, x.h), __builtin_bit_cast(bf16x8, w.h), c, 0, 0, 0);
    else
      return __builtin_amdgcn_mfma_f32_16x16x32_f16(x.h, w.h, c, 0, 0, 0);
  };

  // codes, scales and zeros of the tile in use and of the next one (scales and zeros as loaded).  Codes have the policy of data
  // that is read once also where workgroups for other batch rows read them again: with the default one, one block of batch rows
  // takes 6 % longer, two the same, three and four 1 and 2 % less (geometric means over 13000 random calls).
  uint32_t wr[kSets][R][Fmt::kWords], sr[kSets][R], zr[kSets][R];
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
  // l%16, which holds chunk (l%16) ^ (row%16) of the row's 256 bytes).
  uint32_t copy_off[kCopies];
#pragma unroll
  for (int i = 0; i < kCopies; i++) {
    const int row = 4 * i + q;
    copy_off[i] = m0 + row < a.M ? (uint32_t)(m0 + row) * (uint32_t)a.K * 2u + (r16 ^ (row & 15)) * 16 : x_bytes;
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
  unsigned char* const stage_odd = smem_odd + (kTwo ? wave * kStage : 0);
  const int xrow = ROWS < 16 ? r16 & (ROWS - 1) : r16;
  constexpr int kLoads = kCopies + R * ((MASTER ? master_load_count(BITS) : tile_load_count(BITS)) + (GROUP == -1 ? 0 : ZP ? 2 : 1));
  static_assert(kLoads < 64, "vmcnt counts up to 63");
  // Tile t of the walk (K tile wave + 8 t) in register set `btag`.  `moretag`: with two buffers tile t + 2 is requested
  // (without it, on the last two tiles, set 0 leaves set 1's requests in flight, set 1 none), with one tile t + 1 as soon as
  // the operands are in registers.
  auto tile = [&](int t, auto btag, auto moretag) {
    constexpr int B = decltype(btag)::value;
    constexpr bool kMore = decltype(moretag)::value;
    constexpr int kYounger = kTwo && (kMore || B == 0) ? kLoads : 0;  // requests of the tile behind this one
    const int kb = wave + t * kWaves;
    unsigned char* const buf = kTwo && B == 1 ? stage_odd : stage_even;
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_waitcnt((kYounger & 15) | (7 << 4) | (15 << 8) | ((kYounger >> 4) << 14));
    __builtin_amdgcn_sched_barrier(0);
    Frag xf[4][MB];
#pragma unroll
    for (int j = 0; j < 4; j++)
#pragma unroll
      for (int i = 0; i < MB; i++)
        xf[j][i].v = *reinterpret_cast<const uint4*>(buf + (i * 16 + xrow) * 256 + (((4 * j + q) ^ xrow) * 16));
    __builtin_amdgcn_sched_barrier(0);
    if constexpr (kMore) {
      __builtin_amdgcn_s_waitcnt(15 | (7 << 4) | (0 << 8) | (3 << 14));  // lgkmcnt(0): the buffer is free
      __builtin_amdgcn_sched_barrier(0);
      copy_x(buf, kb + (kTwo ? 2 : 1) * kWaves);
      if constexpr (!kTwo) load_weights(wr[(B + 1) % kSets], sr[(B + 1) % kSets], zr[(B + 1) % kSets], kb + kWaves);
    }
    // (only the last tile of a walk can lie beyond K; its buffer may hold anything)
    if (kMore || kb < a.k_tiles) {
      const float4v zero4 = {0.f, 0.f, 0.f, 0.f};
      float4v off[MB], xs[MB];
#pragma unroll
      for (int i = 0; i < MB; i++) {
        off[i] = zero4;
        xs[i] = zero4;
#pragma unroll
        for (int j = 0; j < 4; j++) {
          if constexpr (!Raw::kCentred) off[i] = mma(xf[j][i], minus, off[i]);
          if constexpr (ZP) xs[i] = mma(xf[j][i], ones, xs[i]);
        }
        if constexpr (ZP && GROUP == -1) xsum[i] += xs[i];
      }
#pragma unroll
      for (int rr = 0; rr < R; rr++) {
        float4v d[MB];
        float z = 0.f;
        if constexpr (ZP && GROUP != -1) z = 128.0f / kMul - storage_to_float((uint16_t)zr[B][rr]) * (1.0f / kMul);
#pragma unroll
        for (int i = 0; i < MB; i++) {
          d[i] = off[i];
          if constexpr (GROUP == -1) {
            d[i] += acc[rr][i];
          } else if constexpr (ZP) {
#pragma unroll
            for (int e = 0; e < 4; e++) d[i][e] = __builtin_fmaf(z, xs[i][e], d[i][e]);
          }
        }
        auto one = [&](auto jtag) {
          constexpr int J = decltype(jtag)::value;
          Frag codes;
          raw.template octet<J>(wr[B][rr], codes.u);
#pragma unroll
          for (int i = 0; i < MB; i++) d[i] = mma(xf[J][i], codes, d[i]);
        };
        one(std::integral_constant<int, 0>{});
        one(std::integral_constant<int, 1>{});
        one(std::integral_constant<int, 2>{});
        one(std::integral_constant<int, 3>{});
        if constexpr (GROUP == -1) {
#pragma unroll
          for (int i = 0; i < MB; i++) acc[rr][i] = d[i];
        } else {
          const float s = storage_to_float((uint16_t)sr[B][rr]);
#pragma unroll
          for (int i = 0; i < MB; i++)
#pragma unroll
            for (int e = 0; e < 4; e++) acc[rr][i][e] = __builtin_fmaf(s, d[i][e], acc[rr][i][e]);
        }
      }
    }
    __builtin_amdgcn_sched_barrier(0);
    if constexpr (kMore && kTwo) load_weights(wr[B], sr[B], zr[B], kb + 2 * kWaves);
  };

  const int walk = (a.k_tiles + kWaves - 1) / kWaves;  // tiles of the longest walk
  using Even = std::integral_constant<int, 0>;
  using Odd = std::integral_constant<int, 1>;
  __builtin_amdgcn_sched_barrier(0);
  copy_x(stage_even, wave);
  load_weights(wr[0], sr[0], zr[0], wave);
  if constexpr (ONE) {
    tile(0, Even{}, std::false_type{});
  } else if constexpr (!kTwo) {
    // (every tile but the last requests the next one, which lies beyond K for the waves with a shorter walk)
    int t = 0;
    for (; t + 2 < walk; t += 2) {
      tile(t, Even{}, std::true_type{});
      tile(t + 1, Odd{}, std::true_type{});
    }
    if (t + 1 < walk) {
      tile(t, Even{}, std::true_type{});
      tile(t + 1, Odd{}, std::false_type{});
    } else {
      tile(t, Even{}, std::false_type{});
    }
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

  if constexpr (GROUP == -1) {  // the row's one scale and zero point
#pragma unroll
    for (int rr = 0; rr < R; rr++) {
      const int rb = rb_first + rr < a.row_blocks ? rb_first + rr : a.row_blocks - 1;
      const float s = storage_to_float(a.scales[(size_t)rb * 16 + r16]);
      const float z = ZP ? 128.0f / kMul - storage_to_float(a.zeros[(size_t)rb * 16 + r16]) * (1.0f / kMul) : 0.f;
#pragma unroll
      for (int i = 0; i < MB; i++)
#pragma unroll
        for (int e = 0; e < 4; e++) {
          if constexpr (ZP) acc[rr][i][e] = __builtin_fmaf(z, xsum[i][e], acc[rr][i][e]);
          // (a sum times scale 0 is +0, as a sum of products with it is)
          acc[rr][i][e] = __builtin_fmaf(s, acc[rr][i][e], 0.f);
        }
    }
  }

  // Infinities and NaN among a row's activations (and bf16 numbers beyond 2^120) have met zero codes, `base` or the zero
  // point with the other sign and left NaN: a wave with such sums forms them again, with dequantised weights as the
  // other kernels do.  The sums of the other rows stay as they are: what a row gives does not depend on its neighbours.
  bool finite = true;
#pragma unroll
  for (int rr = 0; rr < R; rr++)
#pragma unroll
    for (int i = 0; i < MB; i++)
#pragma unroll
      for (int e = 0; e < 4; e++) finite = finite && __builtin_isfinite(acc[rr][i][e]);
  if (__builtin_amdgcn_ballot_w64(!finite) != 0) {
    const typename Fmt::Consts unpack;
    const BufRsrc xres = make_rsrc(a.x, x_bytes);
    uint32_t x_off[MB];
#pragma unroll
    for (int i = 0; i < MB; i++) {
      const int row = m0 + i * 16 + xrow;
      x_off[i] = row < a.M ? (uint32_t)row * (uint32_t)a.K * 2u + q * 16 : x_bytes;
    }
#pragma unroll
    for (int rr = 0; rr < R; rr++) {
      const int rb = rb_first + rr < a.row_blocks ? rb_first + rr : a.row_blocks - 1;
      float4v again[MB];
#pragma unroll
      for (int i = 0; i < MB; i++) again[i] = float4v{0.f, 0.f, 0.f, 0.f};
      for (int kb = wave; kb < a.k_tiles; kb += kWaves) {
        uint32_t w[Fmt::kWords];
        Fmt::load(make_rsrc(a.packed, w_bytes), (uint32_t)rb * rb_bytes + (uint32_t)kb * tile_bytes, lane, w);
        const size_t g = ((size_t)rb * a.G + (GROUP == -1 ? 0 : kb)) * 16 + r16;
        const float s = storage_to_float(a.scales[g]);
        const float z = ZP ? s * (storage_to_float(a.zeros[g]) - 128.0f) : __uint_as_float(opaque_vgpr(0u));
        auto one = [&](auto jtag) {
          constexpr int J = decltype(jtag)::value;
          Frag aw;
          if constexpr (kBf16) {
            dequant_octet_bf16_fmt<Fmt, BITS, J>(w, unpack, s * kMul, z, aw);
          } else {
            const _Float16 s1 = (_Float16)(s * kMul), z1 = (_Float16)z;
            dequant_octet_fmt<Fmt, BITS, J, true>(w, unpack, half2v{z1, z1}, half2v{s1, s1}, aw);
          }
#pragma unroll
          for (int i = 0; i < MB; i++) {
            const u32x4 v = __builtin_amdgcn_raw_buffer_load_b128(xres, x_off[i], (uint32_t)kb * 256u + J * 64u, 0);
            Frag x;
            x.v = make_uint4(v.x, v.y, v.z, v.w);
            again[i] = mma(x, aw, again[i]);
          }
        };
        one(std::integral_constant<int, 0>{});
        one(std::integral_constant<int, 1>{});
        one(std::integral_constant<int, 2>{});
        one(std::integral_constant<int, 3>{});
      }
#pragma unroll
      for (int i = 0; i < MB; i++)
#pragma unroll
        for (int e = 0; e < 4; e++)
          if (!__builtin_isfinite(acc[rr][i][e])) acc[rr][i][e] = again[i][e] * (1.0f / kMul);
    }
  }

  // The waves' sums of every output meet in LDS (over the activation buffers: every wave has to be done with its
  // own first), four batch rows 4q .. 4q+3 of weight row r16 per lane, row block and batch block.
  __builtin_amdgcn_s_waitcnt(0 | (7 << 4) | (0 << 8) | (0 << 14));  // nothing in flight into LDS any more
  __syncthreads();
  float* const red = reinterpret_cast<float*>(smem_even);
#pragma unroll
  for (int rr = 0; rr < R; rr++)
#pragma unroll
    for (int i = 0; i < MB; i++) *reinterpret_cast<float4v*>(red + (((wave * R + rr) * MB + i) * 64 + lane) * 4) = acc[rr][i];
  __syncthreads();
  for (int o = tid; o < R * MB * 256; o += 64 * kWaves) {
    float sum = red[o];
#pragma unroll
    for (int w = 1; w < kWaves; w++) sum += red[w * R * MB * 256 + o];
    const int l = (o >> 2) & 63, ri = o >> 8;
    const int rb = rb_first + ri / MB, m = m0 + (ri % MB) * 16 + 4 * (l >> 4) + (o & 3);
    if (rb < a.row_blocks && m < a.M) a.y[(size_t)m * a.N + (size_t)rb * 16 + (l & 15)] = float_to_storage(sum * kMul);
  }
}

template <int GROUP, bool ZP, int R, int ROWS, bool MASTER, bool ONE>
hipError_t launch_walk(const GemmArgs& a, hipStream_t stream) {
  if constexpr (few_rows_built(kBits, GROUP, kBf16, MASTER, R, ROWS, ONE)) {
    const int n_tiles = (a.row_blocks + R - 1) / R, m_tiles = (a.M + ROWS - 1) / ROWS;
    const dim3 grid(n_tiles * m_tiles), block(64 * kWaves);
    hipLaunchKernelGGL((few_rows_kernel<kBits, GROUP, ZP, R, ROWS, MASTER, ONE>), grid, block, 0, stream, a, n_tiles, m_tiles);
    return hipGetLastError();
  }
  return hipErrorInvalidValue;
}

template <int GROUP, bool ZP, int R, int ROWS, bool MASTER>
hipError_t launch_r(const GemmArgs& a, hipStream_t stream) {
  return a.k_tiles <= kWaves ? launch_walk<GROUP, ZP, R, ROWS, MASTER, true>(a, stream)
                             : launch_walk<GROUP, ZP, R, ROWS, MASTER, false>(a, stream);
}

template <int GROUP, bool ZP, int R, bool MASTER>
hipError_t launch_batch(const GemmArgs& a, int held, hipStream_t stream) {
  switch (held) {
    case 4: return launch_r<GROUP, ZP, R, 4, MASTER>(a, stream);
    case 8: return launch_r<GROUP, ZP, R, 8, MASTER>(a, stream);
    case 16: return launch_r<GROUP, ZP, R, 16, MASTER>(a, stream);
    default: return launch_r<GROUP, ZP, R, 32, MASTER>(a, stream);
  }
}

template <int GROUP, bool ZP, bool MASTER>
hipError_t launch_rows(const GemmArgs& a, int r, int held, hipStream_t s) {
  switch (r) {
    case 1: return launch_batch<GROUP, ZP, 1, MASTER>(a, held, s);
    case 2: return launch_batch<GROUP, ZP, 2, MASTER>(a, held, s);
    case 4: return launch_batch<GROUP, ZP, 4, MASTER>(a, held, s);
    default: return launch_batch<GROUP, ZP, 8, MASTER>(a, held, s);
  }
}

template <int GROUP, bool ZP>
hipError_t launch_storage(const GemmArgs& a, int r, int held, bool master, hipStream_t s) {
  return master ? launch_rows<GROUP, ZP, true>(a, r, held, s) : launch_rows<GROUP, ZP, false>(a, r, held, s);
}

}  // namespace

#define MATGPTQ_CAT2(a, b) a##b
#define MATGPTQ_CAT(a, b) MATGPTQ_CAT2(a, b)
#if MATGPTQ_BF16
#define MATGPTQ_LAUNCH_NAME MATGPTQ_CAT(MATGPTQ_CAT(launch_few_rows_b, MATGPTQ_BITS), _bf16)
#else
#define MATGPTQ_LAUNCH_NAME MATGPTQ_CAT(launch_few_rows_b, MATGPTQ_BITS)
#endif
// Group size 128 or -1.  r: row blocks of 16 weight rows and held: batch rows per workgroup, as few_rows and few_rows_held give
// them; master: `a.packed` holds master-resident bit planes
hipError_t MATGPTQ_LAUNCH_NAME(const GemmArgs& a, int group_size, int r, int held, bool master, hipStream_t stream) {
  const bool zp = a.zeros != nullptr;
  if (group_size == 32) return hipErrorInvalidValue;
  if (group_size == 128)
    return zp ? launch_storage<128, true>(a, r, held, master, stream) : launch_storage<128, false>(a, r, held, master, stream);
  return zp ? launch_storage<-1, true>(a, r, held, master, stream) : launch_storage<-1, false>(a, r, held, master, stream);
}

}  // namespace matgptq
