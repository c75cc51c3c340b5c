// Few-rows kernel (five to thirty-two batch rows): no staging at all.
// Compiled once per bitwidth with -DMATGPTQ_BITS=b.
//
// At these batch sizes a layer is bound by how soon its bytes are requested, and the mid-batch kernel
// (skinny_gfx950.hip) walks a wave's K tiles one after the other, each waiting for the copy of its activations
// into LDS: eight serial trips to memory on a layer of 8192 columns.  Here a wave asks for everything at once.
//
//  * A workgroup of W waves owns R row blocks of 16 weight rows and all of K.  Wave w owns the T consecutive
//    K tiles [(round W + w) T, +T), round = 0, 1, ...; at the top of a round it requests the scales and zeros,
//    the activations and the R T code tiles of the round and then consumes them in request order.
//  * The activations go from global memory straight into the registers of the MFMA operand: lane (r, q) loads
//    the 16 bytes of batch row r, octet quarter q, so the four lanes of a row read 64 contiguous bytes of
//    one cache line and the second half of the line is the next request's.  They are re-read by every
//    workgroup, from L2; R row blocks share one read.  Nothing passes through LDS, no wait but for the loads,
//    no barrier in the loop.  Batch rows beyond M are out of the descriptor's range and cost no traffic.
//  * Weights are dequantised from registers exactly as in the mid-batch and prefill kernels.
//  * The W partial sums meet in LDS once, at the end.
#include <atomic>

#include "tile_format.h"

#ifndef MATGPTQ_BITS
#error "compile with -DMATGPTQ_BITS={2,3,4,6,8}"
#endif

namespace matgptq {

namespace {

constexpr int kBits = MATGPTQ_BITS;

template <int BITS, int GROUP, bool ZP, int T, int R, int MB, int THREADS>
__global__ void __launch_bounds__(THREADS)
few_kernel(const GemmArgs a, const int W) {
  using Fmt = TileFormat<BITS, false>;
  constexpr int GPT = GROUP == 32 ? 4 : 1;         // scales per tile and row
  constexpr int NS = GROUP == -1 ? 1 : T * GPT;    // scale registers per row block and round
  extern __shared__ __align__(16) unsigned char smem[];

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r16 = lane & 15;
  const int q = lane >> 4;
  const int rb0 = blockIdx.x * R;

  constexpr uint32_t tile_bytes = Fmt::kTileBytes;
  const typename Fmt::Consts consts;
  const uint32_t x_bytes = (uint32_t)a.M * (uint32_t)a.K * 2u;
  uint32_t x_off[MB];
#pragma unroll
  for (int i = 0; i < MB; i++) {
    const uint32_t m = (uint32_t)(i * 16 + r16);
    x_off[i] = m < (uint32_t)a.M ? m * (uint32_t)a.K * 2u + q * 16 : x_bytes;
  }

  float4v acc[R][MB];
#pragma unroll
  for (int rr = 0; rr < R; rr++)
#pragma unroll
    for (int i = 0; i < MB; i++) acc[rr][i] = float4v{0.f, 0.f, 0.f, 0.f};

  for (int kt0 = wave * T; kt0 < a.k_tiles; kt0 += W * T) {
    const int left = a.k_tiles - kt0;
    const int nt = left < T ? left : T;  // tiles of this round; what lies past it reads as zero

    uint16_t sv[R][NS], zv[R][NS];
    uint32_t w[R][T][Fmt::kWords];
    half8 xf[T][4][MB];
#pragma unroll
    for (int rr = 0; rr < R; rr++) {
      const bool rows = rb0 + rr < a.row_blocks;
      const uint32_t g0 = (uint32_t)(rb0 + rr) * a.G + (GROUP == -1 ? 0u : (uint32_t)kt0 * GPT);  // first group of the round
      const uint32_t s_end = rows ? (g0 + (GROUP == -1 ? 1u : (uint32_t)nt * GPT)) * 32u : 0u;
      const BufRsrc sr = make_rsrc(a.scales, s_end);
      const BufRsrc zr = make_rsrc(ZP ? a.zeros : a.scales, s_end);
#pragma unroll
      for (int h = 0; h < NS; h++) {
        sv[rr][h] = __builtin_amdgcn_raw_buffer_load_b16(sr, r16 * 2, (g0 + h) * 32u, 0);
        if constexpr (ZP) zv[rr][h] = __builtin_amdgcn_raw_buffer_load_b16(zr, r16 * 2, (g0 + h) * 32u, 0);
        else zv[rr][h] = 0;
      }
    }
#pragma unroll
    for (int i = 0; i < T; i++) {
      const BufRsrc xr = make_rsrc(a.x, i < nt ? x_bytes : 0u);
#pragma unroll
      for (int j = 0; j < 4; j++)
#pragma unroll
        for (int b = 0; b < MB; b++)
          xf[i][j][b] = __builtin_bit_cast(half8, __builtin_amdgcn_raw_buffer_load_b128(
              xr, (int)x_off[b], (int)((uint32_t)(kt0 + i) * 256u + j * 64u), 0));
    }
#pragma unroll
    for (int i = 0; i < T; i++)
#pragma unroll
      for (int rr = 0; rr < R; rr++) {
        const uint32_t t0 = (uint32_t)(rb0 + rr) * a.k_tiles + kt0;
        const BufRsrc wr = make_rsrc(a.packed, rb0 + rr < a.row_blocks ? (t0 + nt) * tile_bytes : 0u);
        Fmt::load(wr, (t0 + i) * tile_bytes, lane, w[rr][i]);
      }
    __builtin_amdgcn_sched_barrier(0);

#pragma unroll
    for (int i = 0; i < T; i++) {
      auto one = [&](auto jtag) {
        constexpr int J = decltype(jtag)::value;
        Frag aw[R];
#pragma unroll
        for (int rr = 0; rr < R; rr++) {
          const int g = GROUP == -1 ? 0 : GROUP == 32 ? i * 4 + J : i;
          if constexpr (kBf16) {
            const float s0 = bf16_bits_to_float(sv[rr][g]);
            const float sm = s0 * (float)(1 << (8 - BITS));
            float sz = 0.f;
            if constexpr (ZP) sz = s0 * (bf16_bits_to_float(zv[rr][g]) - 128.0f);
            dequant_octet_bf16_fmt<Fmt, BITS, J>(w[rr][i], consts, sm, sz, aw[rr]);
          } else {
            // scale * 2^(8-b) and scale * (zero - 128)
            const _Float16 s0 = __builtin_bit_cast(_Float16, sv[rr][g]);
            const _Float16 s1 = (_Float16)((float)s0 * (float)(1 << (8 - BITS)));
            _Float16 z1 = (_Float16)0.f;
            if constexpr (ZP) z1 = s0 * (__builtin_bit_cast(_Float16, zv[rr][g]) - (_Float16)128.0f);
            dequant_octet_fmt<Fmt, BITS, J, ZP>(w[rr][i], consts, half2v{z1, z1}, half2v{s1, s1}, aw[rr]);
          }
        }
#pragma unroll
        for (int b = 0; b < MB; b++)
#pragma unroll
          for (int rr = 0; rr < R; rr++) {
            if constexpr (kBf16)
              acc[rr][b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, aw[rr].h),
                                                                  __builtin_bit_cast(bf16x8, xf[i][J][b]), acc[rr][b], 0, 0, 0);
            else
              acc[rr][b] = __builtin_amdgcn_mfma_f32_16x16x32_f16(aw[rr].h, xf[i][J][b], acc[rr][b], 0, 0, 0);
          }
      };
      one(std::integral_constant<int, 0>{});
      one(std::integral_constant<int, 1>{});
      one(std::integral_constant<int, 2>{});
      one(std::integral_constant<int, 3>{});
    }
  }

  // the W partial sums: red[wave][rr * MB + b][lane]
  float4v* const red = reinterpret_cast<float4v*>(smem);
#pragma unroll
  for (int rr = 0; rr < R; rr++)
#pragma unroll
    for (int b = 0; b < MB; b++) red[((wave * R + rr) * MB + b) * 64 + lane] = acc[rr][b];
  __syncthreads();
  for (int ot = tid; ot < R * MB * 64; ot += 64 * W) {
    float4v sum = red[ot];
    for (int w2 = 1; w2 < W; w2++) sum += red[w2 * R * MB * 64 + ot];
    const int l = ot & 63, ri = ot >> 6;
    const int rb = rb0 + ri / MB;
    const int m = (ri % MB) * 16 + (l & 15);
    if (rb < a.row_blocks && m < a.M) {
      uint16_t o[4];
#pragma unroll
      for (int e = 0; e < 4; e++) o[e] = float_to_storage(sum[e]);
      *reinterpret_cast<uint2*>(a.y + (size_t)m * a.N + (size_t)rb * 16 + 4 * (l >> 4)) =
          make_uint2((uint32_t)o[0] | ((uint32_t)o[1] << 16), (uint32_t)o[2] | ((uint32_t)o[3] << 16));
    }
  }
}

template <int GROUP, bool ZP, int T, int R, int MB, int THREADS>
hipError_t launch_one(const GemmArgs& a, int W, hipStream_t stream) {
  const size_t smem = (size_t)W * R * MB * 1024;
  if (W < 1 || 64 * W > THREADS || a.M > 16 * MB || smem > 64 * 1024) return hipErrorInvalidValue;
  hipLaunchKernelGGL((few_kernel<kBits, GROUP, ZP, T, R, MB, THREADS>), dim3((a.row_blocks + R - 1) / R), dim3(64 * W),
                     smem, stream, a, W);
  return hipGetLastError();
}

template <int GROUP, bool ZP>
hipError_t launch_shape(const GemmArgs& a, int shape, int W, hipStream_t s) {
  switch (shape) {
    case 0: return launch_one<GROUP, ZP, 4, 1, 1, 1024>(a, W, s);
    case 1: return launch_one<GROUP, ZP, 2, 2, 1, 1024>(a, W, s);
    case 2: return launch_one<GROUP, ZP, 4, 2, 1, 512>(a, W, s);
    case 3: return launch_one<GROUP, ZP, 2, 4, 1, 512>(a, W, s);
    case 4: return launch_one<GROUP, ZP, 2, 1, 1, 1024>(a, W, s);
    case 5: return launch_one<GROUP, ZP, 1, 4, 1, 1024>(a, W, s);
    case 6: return launch_one<GROUP, ZP, 2, 2, 2, 512>(a, W, s);
    case 7: return launch_one<GROUP, ZP, 1, 4, 2, 512>(a, W, s);
    case 8: return launch_one<GROUP, ZP, 2, 1, 2, 1024>(a, W, s);
    default: return hipErrorInvalidValue;
  }
}

}  // namespace

#define MATGPTQ_CAT2(a, b) a##b
#define MATGPTQ_CAT(a, b) MATGPTQ_CAT2(a, b)
#if MATGPTQ_BF16
#define MATGPTQ_LAUNCH_NAME MATGPTQ_CAT(MATGPTQ_CAT(launch_few_b, MATGPTQ_BITS), _bf16)
#else
#define MATGPTQ_LAUNCH_NAME MATGPTQ_CAT(launch_few_b, MATGPTQ_BITS)
#endif
// shape: index into the table above; W: waves per workgroup
hipError_t MATGPTQ_LAUNCH_NAME(const GemmArgs& a, int group_size, int shape, int W, hipStream_t stream) {
  const bool zp = a.zeros != nullptr;
  if (group_size == 128) return zp ? launch_shape<128, true>(a, shape, W, stream) : launch_shape<128, false>(a, shape, W, stream);
  if (group_size == 32) return zp ? launch_shape<32, true>(a, shape, W, stream) : launch_shape<32, false>(a, shape, W, stream);
  return zp ? launch_shape<-1, true>(a, shape, W, stream) : launch_shape<-1, false>(a, shape, W, stream);
}

}  // namespace matgptq
