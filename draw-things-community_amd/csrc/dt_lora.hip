// The low-rank branch of a LoRADense in high precision: up(scale * down(float(x))) with fp32 weights, fp32
// intermediate and fp32 accumulation, rounded to fp16 once at the end (Models/LoRA.swift:117-139, highPrecision:
// `denseDown(x.to(.Float32))`, `denseUp(scale * downX).to(of: x)`).  Two GEMMs on the fp32 matrix instructions with
// nothing in common but the rank (4 .. 128): the first is long in K and narrow, the second short in K and writes the
// whole output.  The base projection's epilogue then adds the branch as its `addend`.
#include "dt_common.h"

namespace dt {

typedef uint32_t u32x4_h __attribute__((ext_vector_type(4), aligned(2)));  // (the part reads words at any address)
typedef float float4_a4 __attribute__((ext_vector_type(4), aligned(4)));

struct LoraDownArgs {
  const uint16_t* x;
  int64_t ldx, m, k;
  const float* down;
  int32_t rank;
  float scale;
  float* t;
};

// T[M, rank] = scale * float(X)[M, K] down[rank, K]^T: 16 * MT rows x 16 * RT ranks per 512-thread workgroup, every wave
// the whole block over every eighth stretch of 32 k, straight from memory into registers (lane: row l % 16, k 8 (l / 16)
// .. + 7; the j-th v_mfma_f32_16x16x4_f32 of a stretch takes the lanes' j-th values), their sums added up in LDS.
// Bound by what a compute unit's L1 can have in flight: every workgroup reads all of `down`, and a CU pulls some 25 GB/s
// past its L1.  4608 x 3072, rank 32: 21 us (a 64 x 64 tile with 16-wide K steps through LDS: 235 us).
template <int MT, int RT>
__global__ void __launch_bounds__(512) lora_down_kernel(const LoraDownArgs a) {
  constexpr int NW = 8, RB = 16 * RT, MB = 16 * MT;
  __shared__ float red[NW * MB * (RB + 1)];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int l16 = lane & 15, c = lane >> 4;
  const int64_t m0 = (int64_t)blockIdx.x * MB;
  const int r0 = (int)blockIdx.y * RB;
  const uint16_t* xr[MT];
  const float* dr[RT];
#pragma unroll
  for (int i = 0; i < MT; i++) xr[i] = a.x + (m0 + 16 * i + l16 < a.m ? m0 + 16 * i + l16 : a.m - 1) * a.ldx;
#pragma unroll
  for (int i = 0; i < RT; i++) dr[i] = a.down + (int64_t)(r0 + 16 * i + l16 < a.rank ? r0 + 16 * i + l16 : a.rank - 1) * a.k;

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
    a.t[(m0 + m) * a.rank + r0 + r] = s * a.scale;  // the scale is its own fp32 multiplication, as in the graph
  }
}

struct LoraUpArgs {
  const float* t;
  int64_t m, n;
  const float* up;
  int32_t rank;
  uint16_t* out;
  int64_t ldo;
};

// out[M, N] = fp16(T[M, rank] up[N, rank]^T): 64 x 128 outputs per 256-thread workgroup, a wave 64 x 32 on
// v_mfma_f32_32x32x2_f32.  The operands come straight from memory (lane: row l % 32, ranks 8 (l / 32) .. + 7 of every
// 16; the j-th instruction takes the lanes' j-th values); the result is parked in LDS so that it leaves in whole 16-byte
// pieces of consecutive addresses.  Bound by the output's 28 MB and the fp32 matrix rate: 4608 x 3072, rank 16 / 32 /
// 128: 11 / 20 / 56 us (2-byte stores from the accumulator layout and K steps through LDS: 32 us at rank 32).
__global__ void __launch_bounds__(256) lora_up_kernel(const LoraUpArgs a) {
  constexpr int TM = 64, TN = 128, LDO = TN + 8;
  __shared__ __attribute__((aligned(16))) half_t park[TM * LDO];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int l32 = lane & 31, hi = lane >> 5;
  const int64_t m0 = (int64_t)blockIdx.x * TM, n0 = (int64_t)blockIdx.y * TN;
  const auto row = [](int64_t r, int64_t n) { return r < n ? r : n - 1; };
  const float* src[3] = {a.t + row(m0 + l32, a.m) * a.rank, a.t + row(m0 + 32 + l32, a.m) * a.rank,
                         a.up + row(n0 + wave * 32 + l32, a.n) * a.rank};
  float16_t acc[2];
#pragma unroll
  for (int i = 0; i < 2; i++)
#pragma unroll
    for (int v = 0; v < 16; v++) acc[i][v] = 0.f;
  for (int r0 = 0; r0 < a.rank; r0 += 16) {
    float4_a4 v[3][2];
    if (r0 + 16 <= a.rank) {  // uniform
#pragma unroll
      for (int i = 0; i < 3; i++)
#pragma unroll
        for (int h = 0; h < 2; h++) v[i][h] = *reinterpret_cast<const float4_a4*>(src[i] + r0 + 8 * hi + 4 * h);
    } else {
#pragma unroll
      for (int i = 0; i < 3; i++)
#pragma unroll
        for (int j = 0; j < 8; j++) {
          const bool on = r0 + 8 * hi + j < a.rank;
          const float f = src[i][on ? r0 + 8 * hi + j : 0];
          v[i][j >> 2][j & 3] = on ? f : 0.f;
        }
    }
#pragma unroll
    for (int j = 0; j < 8; j++)
#pragma unroll
      for (int i = 0; i < 2; i++)
        acc[i] = __builtin_amdgcn_mfma_f32_32x32x2f32(v[i][j >> 2][j & 3], v[2][j >> 2][j & 3], acc[i], 0, 0, 0);
  }
  // lane holds column n = l32 of the wave's 32 and rows m = 8 (v / 4) + 4 hi + v % 4 of each block
#pragma unroll
  for (int i = 0; i < 2; i++)
#pragma unroll
    for (int v = 0; v < 16; v++) park[(i * 32 + 8 * (v >> 2) + 4 * hi + (v & 3)) * LDO + wave * 32 + l32] = (half_t)acc[i][v];
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

template <int MT>
static void launch_down(hipStream_t s, const LoraDownArgs& a) {
  const unsigned gx = (unsigned)((a.m + 16 * MT - 1) / (16 * MT));
  if (a.rank <= 16) hipLaunchKernelGGL((lora_down_kernel<MT, 1>), dim3(gx), dim3(512), 0, s, a);
  else if (a.rank <= 32) hipLaunchKernelGGL((lora_down_kernel<MT, 2>), dim3(gx), dim3(512), 0, s, a);
  else hipLaunchKernelGGL((lora_down_kernel<MT, 4>), dim3(gx, (unsigned)((a.rank + 63) / 64)), dim3(512), 0, s, a);
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
  const LoraDownArgs d{X, ldx, M, K, down, rank, scale, T};
  // 32 rows a workgroup halve what is read of `down`, 16 reach twice as many compute units: 16 up to one workgroup per CU
  // (rank 32, 3072 wide, 16 / 32 rows: 512 rows 16.3 / 20.1 us, 4608 rows 30.2 / 20.7; 1280 wide, 1500 rows 8.4 / 11.4)
  if (M > 16 * 256) launch_down<2>(s, d);
  else launch_down<1>(s, d);
  if (const dt_status st = launch_status(); st != DT_OK) return st;
  const LoraUpArgs u{T, M, N, up, rank, out, ldo};
  hipLaunchKernelGGL(lora_up_kernel, dim3((unsigned)((M + 63) / 64), (unsigned)((N + 127) / 128)), dim3(256), 0, s, u);
  return launch_status();
}
