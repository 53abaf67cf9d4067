// The second half of a LoRA layer's low-rank branch, T[M, rank] up[N, rank]^T, as sums in registers: what the Dense epilogue adds
// to its tile, and the kernel of the branch alone.
#pragma once
#include <type_traits>

#include "dt_common.h"

namespace dt {

// T and up of a layer, both fp16 (`rank` 16 or 32, all rows 8-byte aligned) or both fp32 (any rank).
struct DenseLora {
  const void* t;   // [M, rank], scale included, row stride ld_t
  const void* up;  // [N, rank], row stride ld_up; null = no branch
  int64_t ld_t, ld_up;
  int32_t rank;
  int32_t f32;
};

// s[i][j] = sums of features n0 + 16 i .. + 15 (rows: lane holds 4 (lane / 16) .. + 3) and tokens m0 + 16 j .. + 15 (column lane % 16);
// what lies outside reads the last row.  fp16: v_mfma_f32_16x16x16_f16 from rank 0 up, two of which give the same bits as the
// v_mfma_f32_16x16x32_f16 of the tiled kernels does (65536 sums of random operands: none differs; a measurement, which the tests hold,
// and no statement of the instruction's).  KEEP: the rows' addresses stay in registers from step to step (4608 x 3072, rank 128 in fp32, us:
// 57.8 for the kernel of the branch alone, 73.8 without; a Dense epilogue has no room for them).  The operands come straight from memory: they are read once or twice from a cache, and a launch is a few K-tiles long.
template <int TN, int TM, bool KEEP = false>
__device__ __forceinline__ void low_rank_sums(float4_t (&s)[TN][TM], const DenseLora& l, int64_t n0, int64_t n, int64_t m0, int64_t m, int lane) {
  typedef float float4_a4 __attribute__((ext_vector_type(4), aligned(4)));
  typedef half_t half4_t __attribute__((ext_vector_type(4)));
  const auto row = [](int64_t at, int64_t end, int64_t ld) { return (at < end ? at : end - 1) * ld; };
#pragma unroll
  for (int i = 0; i < TN; i++)
#pragma unroll
    for (int j = 0; j < TM; j++) s[i][j] = float4_t{0.f, 0.f, 0.f, 0.f};
  // RS steps of 16 ranks, all of whose operands are asked for at once: a trip to memory takes longer than the multiplications
  const auto steps = [&](auto f32, auto count, int r0) {
    constexpr int RS = decltype(count)::value;
    // (the rows' addresses out of the registers that live across a loop)
    if constexpr (!KEEP) asm volatile("" : "+v"(lane));
    const int l16 = lane & 15, r = r0 + 4 * (lane >> 4);
    if constexpr (!decltype(f32)::value) {
      const half_t *const T = static_cast<const half_t*>(l.t) + r, *const U = static_cast<const half_t*>(l.up) + r;
      half4_t a[RS][TN], b[RS][TM];
#pragma unroll
      for (int k = 0; k < RS; k++) {
#pragma unroll
        for (int j = 0; j < TM; j++) b[k][j] = *reinterpret_cast<const half4_t*>(T + row(m0 + 16 * j + l16, m, l.ld_t) + 16 * k);
#pragma unroll
        for (int i = 0; i < TN; i++) a[k][i] = *reinterpret_cast<const half4_t*>(U + row(n0 + 16 * i + l16, n, l.ld_up) + 16 * k);
      }
#pragma unroll
      for (int k = 0; k < RS; k++)
#pragma unroll
        for (int i = 0; i < TN; i++)
#pragma unroll
          for (int j = 0; j < TM; j++) s[i][j] = __builtin_amdgcn_mfma_f32_16x16x16f16(a[k][i], b[k][j], s[i][j], 0, 0, 0);
    } else {
      // fp32: of every 16 ranks a lane holds 4 quad .. + 3, and the e-th v_mfma_f32_16x16x4_f32 takes the lanes' e-th ones
      const float *const T = static_cast<const float*>(l.t), *const U = static_cast<const float*>(l.up);
      float4_a4 a[RS][TN], b[RS][TM];
#pragma unroll
      for (int k = 0; k < RS; k++) {
        const int rk = r + 16 * k;
        const bool whole = r0 + 16 * k + 16 <= l.rank;  // uniform
        const auto ranks = [&](const float* at) {
          float4_a4 v;
          if (whole) {
            v = *reinterpret_cast<const float4_a4*>(at + rk);
          } else {
#pragma unroll
            for (int e = 0; e < 4; e++) {
              const float f = at[rk + e < l.rank ? rk + e : 0];
              v[e] = rk + e < l.rank ? f : 0.f;
            }
          }
          return v;
        };
#pragma unroll
        for (int j = 0; j < TM; j++) b[k][j] = ranks(T + row(m0 + 16 * j + l16, m, l.ld_t));
#pragma unroll
        for (int i = 0; i < TN; i++) a[k][i] = ranks(U + row(n0 + 16 * i + l16, n, l.ld_up));
      }
#pragma unroll
      for (int k = 0; k < RS; k++)
#pragma unroll
        for (int e = 0; e < 4; e++)
#pragma unroll
          for (int i = 0; i < TN; i++)
#pragma unroll
            for (int j = 0; j < TM; j++) s[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[k][i][e], b[k][j][e], s[i][j], 0, 0, 0);
    }
  };
  int r0 = 0;
  if (l.f32) {
#pragma unroll 1
    for (; r0 + 32 <= l.rank; r0 += 32) steps(std::true_type{}, std::integral_constant<int, 2>{}, r0);
#pragma unroll 1
    for (; r0 < l.rank; r0 += 16) steps(std::true_type{}, std::integral_constant<int, 1>{}, r0);
  } else {
    if (l.rank > 16) steps(std::false_type{}, std::integral_constant<int, 2>{}, 0);
    else steps(std::false_type{}, std::integral_constant<int, 1>{}, 0);
  }
}

}  // namespace dt
