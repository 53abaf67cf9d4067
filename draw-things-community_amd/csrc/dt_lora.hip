// The low-rank branch of a LoRADense: up(scale * down(x)) (Models/LoRA.swift:85-142).  Its first half here, in fp16 and, for a pair
// in high precision (`denseDown(x.to(.Float32))`, `denseUp(scale * downX).to(of: x)`, 117-139), with fp32 weights, intermediate and
// accumulation; the second half is added by the epilogue of the base projection, or for the fp32 branch alone written by a kernel here.
#include <type_traits>

#include "dt_common.h"
#include "dt_lora.h"
#include "dt_low_rank.h"

namespace dt {

typedef uint32_t u32x4_h __attribute__((ext_vector_type(4), aligned(2)));  // (the part reads words at any address)
typedef half_t half4_t __attribute__((ext_vector_type(4)));
typedef float float4_a4 __attribute__((ext_vector_type(4), aligned(4)));

// fp32: T[M, rank] = scale * float(X)[M, K] down[rank, K]^T: 16 * MT rows x 16 * RT ranks per 512-thread workgroup, every wave
// the whole block over every eighth stretch of 32 k, straight from memory into registers (lane: row l % 16, k 8 (l / 16)
// .. + 7; the j-th v_mfma_f32_16x16x4_f32 of a stretch takes the lanes' j-th values), their sums added up in LDS.
// Bound by what a compute unit's L1 can have in flight: every workgroup reads all of `down`, and a CU pulls some 25 GB/s
// past its L1.  4608 x 3072, rank 32: 21 us (a 64 x 64 tile with 16-wide K steps through LDS: 235 us).
template <int MT, int RT>
constexpr int lora_down_f32_lds = 8 * 16 * MT * (16 * RT + 1) * 4;
template <int MT, int RT>
__device__ __forceinline__ void lora_down_f32(const LoraDownArgs& a, int block_m, int block_r, unsigned char* smem) {
  constexpr int NW = 8, RB = 16 * RT, MB = 16 * MT;
  float* const red = reinterpret_cast<float*>(smem);
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int l16 = lane & 15, c = lane >> 4;
  const int64_t m0 = (int64_t)block_m * MB;
  const int r0 = block_r * RB;
  const uint16_t* xr[MT];
  const float* dr[RT];
#pragma unroll
  for (int i = 0; i < MT; i++) xr[i] = a.x + (m0 + 16 * i + l16 < a.m ? m0 + 16 * i + l16 : a.m - 1) * a.ldx;
#pragma unroll
  for (int i = 0; i < RT; i++) dr[i] = static_cast<const float*>(a.down) + (int64_t)(r0 + 16 * i + l16 < a.rank ? r0 + 16 * i + l16 : a.rank - 1) * a.k;

  float4_t acc[MT][RT];
#pragma unroll
  for (int i = 0; i < MT; i++)
#pragma unroll
    for (int j = 0; j < RT; j++) acc[i][j] = float4_t{0.f, 0.f, 0.f, 0.f};
  u32x4_h xv[2][MT];
  float4_a4 dv[2][RT][2];
  const int64_t n_step = a.k / 32;  // whole stretches
  auto fetch = [&](int buf, int64_t step) {
    const int64_t k0 = 32 * step + 8 * c;
#pragma unroll
    for (int i = 0; i < MT; i++) xv[buf][i] = *reinterpret_cast<const u32x4_h*>(xr[i] + k0);
#pragma unroll
    for (int i = 0; i < RT; i++)
#pragma unroll
      for (int h = 0; h < 2; h++) dv[buf][i][h] = *reinterpret_cast<const float4_a4*>(dr[i] + k0 + 4 * h);
  };
  auto multiply = [&](int buf) {
#pragma unroll
    for (int j = 0; j < 8; j++)
#pragma unroll
      for (int i = 0; i < MT; i++) {
        const float x = (float)bits_to_half((uint16_t)(xv[buf][i][j >> 1] >> (16 * (j & 1))));
#pragma unroll
        for (int r = 0; r < RT; r++)
          acc[i][r] = __builtin_amdgcn_mfma_f32_16x16x4f32(x, dv[buf][r][j >> 2][j & 3], acc[i][r], 0, 0, 0);
      }
  };
  if (wave < n_step) fetch(0, wave);
  for (int64_t step = wave; step < n_step; step += 2 * NW) {
    if (step + NW < n_step) fetch(1, step + NW);
    multiply(0);
    if (step + NW < n_step) {
      if (step + 2 * NW < n_step) fetch(0, step + 2 * NW);
      multiply(1);
    }
  }
  if (a.k % 32 != 0 && wave == (int)(n_step % NW)) {  // the rest of K, element by element
    const int64_t k0 = 32 * n_step + 8 * c;
#pragma unroll
    for (int i = 0; i < MT; i++) {
      xv[0][i] = u32x4_h{0, 0, 0, 0};
#pragma unroll
      for (int j = 0; j < 8; j++)
        if (k0 + j < a.k) xv[0][i][j >> 1] |= (uint32_t)xr[i][k0 + j] << (16 * (j & 1));
    }
#pragma unroll
    for (int i = 0; i < RT; i++)
#pragma unroll
      for (int j = 0; j < 8; j++) dv[0][i][j >> 2][j & 3] = k0 + j < a.k ? dr[i][k0 + j] : 0.f;
    multiply(0);
  }
  // lane holds rank l16 and rows 4 c .. 4 c + 3 of each block
#pragma unroll
  for (int i = 0; i < MT; i++)
#pragma unroll
    for (int r = 0; r < RT; r++)
#pragma unroll
      for (int v = 0; v < 4; v++) red[(wave * MB + 16 * i + 4 * c + v) * (RB + 1) + 16 * r + l16] = acc[i][r][v];
  __syncthreads();
  for (int i = tid; i < MB * RB; i += 512) {
    const int m = i / RB, r = i % RB;
    if (m0 + m >= a.m || r0 + r >= a.rank) continue;
    float s = 0.f;
#pragma unroll
    for (int p = 0; p < NW; p++) s += red[(p * MB + m) * (RB + 1) + r];
    static_cast<float*>(a.t)[(m0 + m) * a.rank + r0 + r] = s * a.scale;  // the scale is its own fp32 multiplication, as in the graph
  }
}

// fp16: 16 * MT rows and 16 * RT ranks a workgroup.  The sums have to be those of the tiled kernels bit for bit, which go through K in steps of
// 32, so K cannot be shared out between waves whose sums are added up; instead the sums travel from wave to wave through LDS, and
// each adds the S steps that it holds the operands of (lane: row l % 16, k 8 (l / 16) .. + 7 of every step), which it asked for a round of
// the NW waves before.
// (us, the whole layer, 4608 x 3072 -> 3072 q6p, rank 16: one wave over the whole of K with twelve steps in flight 110, this form with 16 rows a
// workgroup 102, with 32 rows 96; twelve steps a turn instead of six 107.)
// Bound by what a compute unit's L1 can have in flight, as above.  K a multiple of 64, X and down rows 16-byte aligned, rank a multiple of 16.
template <int MT, int RT>
constexpr int lora_down_f16_lds = MT * RT * 256 * 4;
template <int MT, int RT>
__device__ __forceinline__ void lora_down_f16(const LoraDownArgs& a, int block_m, int block_r, unsigned char* smem) {
  constexpr int NW = 8, S = MT + RT <= 3 ? 6 : 4;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), l16 = lane & 15, c = lane >> 4;
  float* const sums = reinterpret_cast<float*>(smem) + lane;  // [MT * RT][4][64 lanes]
  const int64_t m = (int64_t)block_m * 16 * MT + l16;
  const int r0 = block_r * 16 * RT;
  const half_t *x[MT], *w[RT];
#pragma unroll
  for (int t = 0; t < MT; t++) x[t] = reinterpret_cast<const half_t*>(a.x) + (m + 16 * t < a.m ? m + 16 * t : a.m - 1) * a.ldx + 8 * c;
#pragma unroll
  for (int r = 0; r < RT; r++) w[r] = static_cast<const half_t*>(a.down) + (int64_t)(r0 + 16 * r < a.rank ? r0 + 16 * r + l16 : l16) * a.k + 8 * c;
  const int n_step = (int)(a.k / 32), rounds = (n_step + NW * S - 1) / (NW * S);
  half8_t xv[MT][S], wv[RT][S];
  // (past the end of K: the last step again, which nothing uses)
  auto fetch = [&](int round) {
#pragma unroll
    for (int i = 0; i < S; i++) {
      const int step = (round * NW + wave) * S + i;
      const int64_t k0 = 32 * (int64_t)(step < n_step ? step : n_step - 1);
#pragma unroll
      for (int t = 0; t < MT; t++) xv[t][i] = *reinterpret_cast<const half8_t*>(x[t] + k0);
#pragma unroll
      for (int r = 0; r < RT; r++) wv[r][i] = *reinterpret_cast<const half8_t*>(w[r] + k0);
    }
  };
  auto turn = [&](int round) {
    float4_t acc[MT * RT];
#pragma unroll
    for (int r = 0; r < MT * RT; r++)
#pragma unroll
      for (int e = 0; e < 4; e++) acc[r][e] = sums[r * 256 + e * 64];
    const int left = n_step - (round * NW + wave) * S;  // an even number
#pragma unroll
    for (int i = 0; i < S; i += 2)
      if (i < left) {  // uniform
#pragma unroll
        for (int h = 0; h < 2; h++)
#pragma unroll
          for (int r = 0; r < MT * RT; r++)
            acc[r] = __builtin_amdgcn_mfma_f32_16x16x32_f16(wv[r % RT][i + h], xv[r / RT][i + h], acc[r], 0, 0, 0);
      }
#pragma unroll
    for (int r = 0; r < MT * RT; r++)
#pragma unroll
      for (int e = 0; e < 4; e++) sums[r * 256 + e * 64] = acc[r][e];
  };
  if (wave * S < n_step) fetch(0);
  if (wave == 0)
#pragma unroll
    for (int r = 0; r < MT * RT; r++)
#pragma unroll
      for (int e = 0; e < 4; e++) sums[r * 256 + e * 64] = 0.f;
  for (int round = 0; round + 1 < rounds; round++) {  // (every wave comes to NW barriers a round)
    for (int i = 0; i < wave; i++) __syncthreads();
    turn(round);
    fetch(round + 1);
    for (int i = wave; i < NW; i++) __syncthreads();
  }
  const int last = (n_step - (rounds - 1) * NW * S + S - 1) / S;  // waves with a share of the last round
  for (int i = 0; i < last; i++) {
    if (i == wave) turn(rounds - 1);
    __syncthreads();
  }
  for (int r = wave; r < MT * RT; r += NW) {
    const int64_t mr = m + 16 * (r / RT);
    const int rank = r0 + 16 * (r % RT);
    if (rank >= a.rank || mr >= a.m) continue;
    half4_t v;
#pragma unroll
    for (int e = 0; e < 4; e++) {
      v[e] = (half_t)sums[r * 256 + e * 64];
      if (a.scale != 1.0f) v[e] = (half_t)((float)v[e] * a.scale);
    }
    *reinterpret_cast<half4_t*>(static_cast<half_t*>(a.t) + mr * a.rank + rank + 4 * c) = v;
  }
}

// A layer's down projection by the first `down_blocks` workgroups; COPIES: palettized weights are written out as fp16 by those behind
// them, on the compute units that the few workgroups of the first leave idle.
struct LoraCopies {
  DepalettizeMany d;
  int32_t qbits;
};
struct NoCopies {};
template <bool F32, int MT, int RT, typename COPIES>
__global__ void __launch_bounds__(512, (F32 ? 2 : 4)) lora_down_kernel(const LoraDownArgs a, const int blocks_m, const int down_blocks, const COPIES c) {
  constexpr bool kCopies = std::is_same<COPIES, LoraCopies>::value;
  constexpr int kDown = F32 ? lora_down_f32_lds<MT, RT> : lora_down_f16_lds<MT, RT>, kCopy = kCopies ? depalettize_lds(8, kLoraCopyGranules) : 0;
  constexpr int kLds = kDown > kCopy ? kDown : kCopy;
  __shared__ __attribute__((aligned(16))) unsigned char smem[kLds];
  if (!kCopies || (int)blockIdx.x < down_blocks) {
    if constexpr (F32) lora_down_f32<MT, RT>(a, (int)blockIdx.x % blocks_m, (int)blockIdx.x / blocks_m, smem);
    else lora_down_f16<MT, RT>(a, (int)blockIdx.x % blocks_m, (int)blockIdx.x / blocks_m, smem);
    return;
  }
  if constexpr (kCopies) {
    const int tile = (int)blockIdx.x - down_blocks;
    if (tile == 0)
      for (int i = threadIdx.x; i < c.d.n_counters; i += 512) c.d.counters[i] = 0;
    const auto& w = c.d.w[0];
    switch (c.qbits) {
      case 4: depalettize_tile<4, kLoraCopyGranules>(w.packed, c.d.nib, w.n_granules, tile, w.out, smem); break;
      case 5: depalettize_tile<5, kLoraCopyGranules>(w.packed, c.d.nib, w.n_granules, tile, w.out, smem); break;
      case 6: depalettize_tile<6, kLoraCopyGranules>(w.packed, c.d.nib, w.n_granules, tile, w.out, smem); break;
      case 7: depalettize_tile<7, kLoraCopyGranules>(w.packed, c.d.nib, w.n_granules, tile, w.out, smem); break;
      default: depalettize_tile<8, kLoraCopyGranules>(w.packed, c.d.nib, w.n_granules, tile, w.out, smem); break;
    }
  }
}

struct LoraUpArgs {
  DenseLora l;
  int64_t m, n;
  uint16_t* out;
  int64_t ldo;
};

// out[M, N] = fp16(T[M, rank] up[N, rank]^T): 64 x 128 outputs per 256-thread workgroup, a wave 64 x 32 (low_rank_sums); the result
// is parked in LDS so that it leaves in whole 16-byte pieces of consecutive addresses.  Bound by the output's 28 MB and the fp32 matrix
// rate (2-byte stores from the accumulator layout and K steps through LDS: 32 us).
__global__ void __launch_bounds__(256) lora_up_kernel(const LoraUpArgs a) {
  constexpr int TM = 64, TN = 128, LDO = TN + 8;
  __shared__ __attribute__((aligned(16))) half_t park[TM * LDO];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int64_t m0 = (int64_t)blockIdx.x * TM, n0 = (int64_t)blockIdx.y * TN;
  float4_t acc[2][4];
  low_rank_sums<2, 4, true>(acc, a.l, n0 + wave * 32, a.n, m0, a.m, lane);
#pragma unroll
  for (int i = 0; i < 2; i++)
#pragma unroll
    for (int j = 0; j < 4; j++)
      *reinterpret_cast<half4_t*>(park + (j * 16 + (lane & 15)) * LDO + wave * 32 + i * 16 + 4 * (lane >> 4)) =
          half4_t{(half_t)acc[i][j][0], (half_t)acc[i][j][1], (half_t)acc[i][j][2], (half_t)acc[i][j][3]};
  __syncthreads();
  const bool vec = a.ldo % 8 == 0 && (reinterpret_cast<uintptr_t>(a.out) & 15) == 0;
#pragma unroll
  for (int p = 0; p < TM * TN / 8 / 256; p++) {
    const int r = (p * 256 + tid) / (TN / 8), ch = tid % (TN / 8);
    const int64_t m = m0 + r, n = n0 + 8 * ch;
    if (m >= a.m || n >= a.n) continue;
    const uint4_t o = *reinterpret_cast<const uint4_t*>(park + r * LDO + 8 * ch);
    uint16_t* dst = a.out + m * a.ldo + n;
    if (vec && n + 8 <= a.n) {
      *reinterpret_cast<uint4_t*>(dst) = o;
    } else {
#pragma unroll
      for (int e = 0; e < 8; e++)
        if (n + e < a.n) dst[e] = (uint16_t)(o[e >> 1] >> (16 * (e & 1)));
    }
  }
}

// Rows (16 MT) and ranks (16 RT) of a workgroup, handed to run(F32, MT, RT, blocks of rows, blocks): the shape for which a compute unit
// reads least.  A step of 32 k takes one read for 16 rows of X and one, in fp32 two, for 16 ranks of `down`; what several
// workgroups on a compute unit read adds up.  (us, the whole layer, all ranks up to 64 in a workgroup / by this rule, rank 32 in fp16: 4608 x 3072 -> 3072 q6p 106 / 101, 1376 x
// 3072 -> 3072 q8p 57 / 54, 512 x 3072 -> 3072 q6p 42 / 38; rank 64 in fp32: 141 / 141, 82 / 70, 62 / 46.)
template <typename F>
static dt_status with_down_shape(const LoraDownArgs& a, const F& run) {
  using std::integral_constant;
  int MT = 1, RT = 1;
  int64_t bm = 0, br = 0, least = INT64_MAX;
  for (int mt = 1; mt <= 2; mt++)
    for (int rt = 1; rt <= (a.f32 ? 4 : 2); rt *= 2) {  // (fp16: ranks up to 32)
      const int64_t m = (a.m + 16 * mt - 1) / (16 * mt), r = (a.rank + 16 * rt - 1) / (16 * rt);
      const int64_t reads = (mt + (a.f32 ? 2 : 1) * rt) * ((m * r + 255) / 256);
      if (reads < least) {
        least = reads;
        bm = m, br = r, MT = mt, RT = rt;
      }
    }
  if (bm * br > 0x3fffffff) return DT_NO_KERNEL;
  const int blocks_m = (int)bm, blocks = (int)(bm * br);
  const auto ranks = [&](auto f32, auto mt) {
    if (RT == 1) run(f32, mt, integral_constant<int, 1>{}, blocks_m, blocks);
    else if (RT == 2) run(f32, mt, integral_constant<int, 2>{}, blocks_m, blocks);
    else if constexpr (decltype(f32)::value) run(f32, mt, integral_constant<int, 4>{}, blocks_m, blocks);
  };
  const auto rows = [&](auto f32) {
    if (MT == 2) ranks(f32, integral_constant<int, 2>{});
    else ranks(f32, integral_constant<int, 1>{});
  };
  if (a.f32) rows(std::true_type{});
  else rows(std::false_type{});
  return launch_status();
}

dt_status lora_down_launch(hipStream_t s, const LoraDownArgs& a) {
  return with_down_shape(a, [&](auto f32, auto mt, auto rt, int blocks_m, int blocks) {
    constexpr bool F32 = decltype(f32)::value;
    constexpr int MT = decltype(mt)::value, RT = decltype(rt)::value;
    hipLaunchKernelGGL((lora_down_kernel<F32, MT, RT, NoCopies>), dim3((unsigned)blocks), dim3(512), 0, s, a, blocks_m, blocks, NoCopies{});
  });
}

dt_status lora_down_copies_launch(hipStream_t s, const LoraDownArgs& a, int qbits, const DepalettizeMany& d, int tiles) {
  const LoraCopies c{d, qbits};
  return with_down_shape(a, [&](auto f32, auto mt, auto rt, int blocks_m, int blocks) {
    constexpr bool F32 = decltype(f32)::value;
    constexpr int MT = decltype(mt)::value, RT = decltype(rt)::value;
    hipLaunchKernelGGL((lora_down_kernel<F32, MT, RT, LoraCopies>), dim3((unsigned)(blocks + tiles)), dim3(512), 0, s, a, blocks_m, blocks, c);
  });
}

}  // namespace dt

DT_EXPORT dt_status dt_lora_branch_f32_f16(dt_stream stream, int64_t M, int64_t K, const uint16_t* X, int64_t ldx,
                                           const float* down, int32_t rank, const float* up, int64_t N, float scale,
                                           float* T, uint16_t* out, int64_t ldo) {
  using namespace dt;
  if (M < 0 || K <= 0 || rank <= 0 || N <= 0 || !down || !up) return DT_INVALID;
  if (M == 0) return DT_OK;
  if (!X || !T || !out || ldx < K || ldo < N) return DT_INVALID;
  if ((reinterpret_cast<uintptr_t>(X) & 1) || (reinterpret_cast<uintptr_t>(out) & 1) || (reinterpret_cast<uintptr_t>(T) & 3) ||
      (reinterpret_cast<uintptr_t>(down) & 3) || (reinterpret_cast<uintptr_t>(up) & 3))
    return DT_INVALID;
  if (!(scale == scale) || scale - scale != 0.f) return DT_INVALID;
  if ((M + 15) / 16 > 0x7fffffff || (N + 127) / 128 > 65535 || (rank + 63) / 64 > 65535) return DT_NO_KERNEL;
  if (const dt_status ready = device_ready(); ready != DT_OK) return ready;
  hipStream_t s = as_stream(stream);
  if (const dt_status st = lora_down_launch(s, LoraDownArgs{X, ldx, M, K, down, rank, 1, scale, T}); st != DT_OK) return st;
  const LoraUpArgs u{DenseLora{T, up, rank, rank, rank, 1}, M, N, out, ldo};
  hipLaunchKernelGGL(lora_up_kernel, dim3((unsigned)((M + 63) / 64), (unsigned)((N + 127) / 128)), dim3(256), 0, s, u);
  return launch_status();
}
