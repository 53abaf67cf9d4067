// K4: LayerNorm(elementwiseAffine: false) over the last axis of an fp32 residual
// stream followed by the adaLN modulation, fp16 out -- the op in front of every
// Dense of a DiT block.  HBM-bound: 4 bytes read and 2 written per element.
// One wave per row; the row stays in registers between the mean, the variance
// and the output pass, so memory is touched once.
#include <type_traits>

#include "dt_common.h"

namespace dt {

__device__ __forceinline__ float wave_sum64(float v) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
  return v;
}

__device__ __forceinline__ float round16(float v) { return round_f16(v); }

// One normalised value through the modulation (sc, sh already widened to float).
//   DT_MOD_F16: fp16(fp16(fp16(n) * scale) + shift), scale and shift fp16
//   DT_MOD_F32: fp16(n * (scale + 1) + shift), scale and shift fp32
//   DT_MOD_AFFINE_F32: fp16(n * scale + shift), scale and shift fp32
template <int MOD>
__device__ __forceinline__ uint16_t modulate(float n, bool has_scale, float sc, bool has_shift, float sh) {
  if constexpr (MOD == DT_MOD_F16) {
    n = round16(n);
    if (has_scale) n = round16(n * sc);
    if (has_shift) n = round16(n + sh);
  } else {
    if (has_scale) n = n * (MOD == DT_MOD_F32 ? sc + 1.0f : sc);
    if (has_shift) n = n + sh;
  }
  return half_to_bits((half_t)n);
}

template <int MOD>
__device__ __forceinline__ float mod_at(const void* p, int64_t c) {
  if constexpr (MOD == DT_MOD_F16) return (float)bits_to_half(static_cast<const uint16_t*>(p)[c]);
  else return static_cast<const float*>(p)[c];
}
// four consecutive values as they lie in memory, and widened
template <int MOD>
using Mod4 = std::conditional_t<MOD == DT_MOD_F16, uint2_t, float4_t>;
template <int MOD>
__device__ __forceinline__ void widen4(const Mod4<MOD>& t, float (&o)[4]) {
  if constexpr (MOD == DT_MOD_F16) {
    o[0] = (float)bits_to_half((uint16_t)t[0]); o[1] = (float)bits_to_half((uint16_t)(t[0] >> 16));
    o[2] = (float)bits_to_half((uint16_t)t[1]); o[3] = (float)bits_to_half((uint16_t)(t[1] >> 16));
  } else {
    o[0] = t[0]; o[1] = t[1]; o[2] = t[2]; o[3] = t[3];
  }
}

struct AdaLnArgs {
  const float* x;
  int64_t ldx;
  int64_t m, c;
  const void* scale;
  const void* shift;
  float eps;
  uint16_t* y;
  int64_t ldy;
};

// Rows of (NV - 2) * 256 + 4 .. NV * 256 elements, C % 4 == 0, 16-byte aligned rows: lane l
// holds the float4 at element 256 i + 4 l of every 256-element chunk i.  Only in the last two chunks can a lane lie past
// the row's end; it then reads the row's first chunk and drops it: behind a test of their own, the chunks' loads (and the
// scale's and shift's, two chunks ahead of their use here) were each waited for before the next went out, 20 us for
// however few rows.  NV goes in steps of two because chunks past the end cost what the others do, and the tests registers:
// in steps of 4, 12 beyond 20, with a test for every chunk, fp32 modulation of 8700 rows took, us, 4608 wide 55.2 (here
// 42.9), 5120 63.2 (48.1, 5.6 TB/s), 6144 88.2 (72.8); 512 rows of 5120 10.0 (7.4).
template <int NV, int MOD>
__global__ void __launch_bounds__(256, NV <= 20 ? 3 : 2) adaln_rows_kernel(const AdaLnArgs a) {
  const int lane = threadIdx.x & 63;
  const int64_t row = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
  if (row >= a.m) return;
  const float* xr = a.x + row * a.ldx;
  uint16_t* yr = a.y + row * a.ldy;
  const int c = (int)a.c;
  float4_t v[NV];
#pragma unroll
  for (int i = 0; i < NV; i++) {
    const int e = i * 256 + lane * 4;
    v[i] = *reinterpret_cast<const float4_t*>(xr + (i < NV - 2 || e < c ? e : 0));
  }
  float s = 0.f;
#pragma unroll
  for (int i = 0; i < NV; i++) {
    if (i >= NV - 2 && i * 256 + lane * 4 >= c) v[i] = float4_t{0.f, 0.f, 0.f, 0.f};
    s += (v[i][0] + v[i][1]) + (v[i][2] + v[i][3]);
  }
  const float mean = wave_sum64(s) / (float)c;
  float q = 0.f;
#pragma unroll
  for (int i = 0; i < NV; i++)
#pragma unroll
    for (int j = 0; j < 4; j++) {
      v[i][j] = i < NV - 2 || i * 256 + lane * 4 < c ? v[i][j] - mean : 0.f;
      q += v[i][j] * v[i][j];
    }
  const float inv = 1.0f / sqrtf(wave_sum64(q) / (float)c + a.eps);
  constexpr int G = 2;  // chunks whose scale and shift are fetched together, one group ahead
  using Raw = Mod4<MOD>;
  Raw sc[2][G], sh[2][G];
  auto fetch = [&](int buf, int i0) {
#pragma unroll
    for (int k = 0; k < G; k++) {
      const int e = (i0 + k) * 256 + lane * 4, ec = i0 + k < NV - 2 || e < c ? e : 0;
      constexpr int W = MOD == DT_MOD_F16 ? 2 : 4;
      if (a.scale) sc[buf][k] = *reinterpret_cast<const Raw*>(static_cast<const char*>(a.scale) + ec * W);
      if (a.shift) sh[buf][k] = *reinterpret_cast<const Raw*>(static_cast<const char*>(a.shift) + ec * W);
    }
  };
  fetch(0, 0);
#pragma unroll
  for (int i = 0; i < NV; i++) {
    const int buf = i / G % 2, k = i % G;
    if (k == 0 && i + G < NV) fetch(buf ^ 1, i + G);
    const int e = i * 256 + lane * 4;
    uint16_t o[4];
    float fs[4] = {0.f, 0.f, 0.f, 0.f}, ft[4] = {0.f, 0.f, 0.f, 0.f};
    if (a.scale) widen4<MOD>(sc[buf][k], fs);
    if (a.shift) widen4<MOD>(sh[buf][k], ft);
#pragma unroll
    for (int j = 0; j < 4; j++)
      o[j] = modulate<MOD>(v[i][j] * inv, a.scale != nullptr, fs[j], a.shift != nullptr, ft[j]);
    if (i < NV - 2 || e < c)
      *reinterpret_cast<uint2_t*>(yr + e) =
          uint2_t{(uint32_t)o[0] | ((uint32_t)o[1] << 16), (uint32_t)o[2] | ((uint32_t)o[3] << 16)};
  }
}

// Any width and alignment: three passes over the row (it stays in cache), scalar accesses.
template <int MOD>
__global__ void __launch_bounds__(256) adaln_generic_kernel(const AdaLnArgs a) {
  const int lane = threadIdx.x & 63;
  const int64_t row = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
  if (row >= a.m) return;
  const float* xr = a.x + row * a.ldx;
  uint16_t* yr = a.y + row * a.ldy;
  float s = 0.f;
  for (int64_t e = lane; e < a.c; e += 64) s += xr[e];
  const float mean = wave_sum64(s) / (float)a.c;
  float q = 0.f;
  for (int64_t e = lane; e < a.c; e += 64) {
    const float d = xr[e] - mean;
    q += d * d;
  }
  const float inv = 1.0f / sqrtf(wave_sum64(q) / (float)a.c + a.eps);
  for (int64_t e = lane; e < a.c; e += 64)
    yr[e] = modulate<MOD>((xr[e] - mean) * inv, a.scale != nullptr, a.scale ? mod_at<MOD>(a.scale, e) : 0.f,
                          a.shift != nullptr, a.shift ? mod_at<MOD>(a.shift, e) : 0.f);
}

// fp16 rows with an elementwise affine weight and bias (fp16), fp16 out: lane l holds the 8 halfs at
// element 512 i + 8 l of every 512-element chunk i.  C % 8 == 0, 16-byte aligned rows, C <= NV * 512.
struct LayerNorm16Args {
  const uint16_t* x;
  int64_t ldx;
  int64_t m, c;
  const uint16_t* gamma;
  const uint16_t* beta;
  float eps;
  uint16_t* y;
  int64_t ldy;
};

__device__ __forceinline__ void unpack8(const uint4_t r, float (&o)[8]) {
#pragma unroll
  for (int q = 0; q < 4; q++) {
    o[2 * q] = (float)bits_to_half((uint16_t)r[q]);
    o[2 * q + 1] = (float)bits_to_half((uint16_t)(r[q] >> 16));
  }
}

template <int NV>
__global__ void __launch_bounds__(256) layernorm16_rows_kernel(const LayerNorm16Args a) {
  const int lane = threadIdx.x & 63;
  const int64_t row = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
  if (row >= a.m) return;
  const uint16_t* xr = a.x + row * a.ldx;
  uint16_t* yr = a.y + row * a.ldy;
  const int c = (int)a.c;
  float v[NV][8];
  float s = 0.f;
#pragma unroll
  for (int i = 0; i < NV; i++) {
    const int e = i * 512 + lane * 8;
    uint4_t r = {0u, 0u, 0u, 0u};
    if (e < c) r = *reinterpret_cast<const uint4_t*>(xr + e);
    unpack8(r, v[i]);
#pragma unroll
    for (int j = 0; j < 8; j++) s += v[i][j];
  }
  const float mean = wave_sum64(s) / (float)c;
  float q = 0.f;
#pragma unroll
  for (int i = 0; i < NV; i++) {
    if (i * 512 + lane * 8 < c) {
#pragma unroll
      for (int j = 0; j < 8; j++) {
        v[i][j] -= mean;
        q += v[i][j] * v[i][j];
      }
    }
  }
  const float inv = 1.0f / sqrtf(wave_sum64(q) / (float)c + a.eps);
#pragma unroll
  for (int i = 0; i < NV; i++) {
    const int e = i * 512 + lane * 8;
    if (e < c) {
      float g[8] = {1.f, 1.f, 1.f, 1.f, 1.f, 1.f, 1.f, 1.f}, b[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
      if (a.gamma) unpack8(*reinterpret_cast<const uint4_t*>(a.gamma + e), g);
      if (a.beta) unpack8(*reinterpret_cast<const uint4_t*>(a.beta + e), b);
      uint32_t o[4];
#pragma unroll
      for (int p = 0; p < 4; p++) {
        const uint16_t lo = half_to_bits((half_t)(v[i][2 * p] * inv * g[2 * p] + b[2 * p]));
        const uint16_t hi = half_to_bits((half_t)(v[i][2 * p + 1] * inv * g[2 * p + 1] + b[2 * p + 1]));
        o[p] = (uint32_t)lo | ((uint32_t)hi << 16);
      }
      *reinterpret_cast<uint4_t*>(yr + e) = uint4_t{o[0], o[1], o[2], o[3]};
    }
  }
}

// any width and alignment
__global__ void __launch_bounds__(256) layernorm16_generic_kernel(const LayerNorm16Args a) {
  const int lane = threadIdx.x & 63;
  const int64_t row = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
  if (row >= a.m) return;
  const uint16_t* xr = a.x + row * a.ldx;
  uint16_t* yr = a.y + row * a.ldy;
  float s = 0.f;
  for (int64_t e = lane; e < a.c; e += 64) s += (float)bits_to_half(xr[e]);
  const float mean = wave_sum64(s) / (float)a.c;
  float q = 0.f;
  for (int64_t e = lane; e < a.c; e += 64) {
    const float d = (float)bits_to_half(xr[e]) - mean;
    q += d * d;
  }
  const float inv = 1.0f / sqrtf(wave_sum64(q) / (float)a.c + a.eps);
  for (int64_t e = lane; e < a.c; e += 64) {
    const float n = ((float)bits_to_half(xr[e]) - mean) * inv;
    const float g = a.gamma ? (float)bits_to_half(a.gamma[e]) : 1.f, b = a.beta ? (float)bits_to_half(a.beta[e]) : 0.f;
    yr[e] = half_to_bits((half_t)(n * g + b));
  }
}

// The instantiation for a row of `nv` chunks.
template <int NV, int MOD>
static void launch_adaln_rows(hipStream_t s, const AdaLnArgs& a, int nv) {
  if constexpr (NV < 32)
    if (nv > NV) return launch_adaln_rows<NV + 2, MOD>(s, a, nv);
  hipLaunchKernelGGL((adaln_rows_kernel<NV, MOD>), dim3((unsigned)((a.m + 3) / 4)), dim3(256), 0, s, a);
}

template <int MOD>
static void launch_adaln(hipStream_t s, const AdaLnArgs& a, bool vec) {
  if (vec && a.c <= 32 * 256) launch_adaln_rows<2, MOD>(s, a, (int)((a.c + 255) / 256));
  else hipLaunchKernelGGL((adaln_generic_kernel<MOD>), dim3((unsigned)((a.m + 3) / 4)), dim3(256), 0, s, a);
}

}  // namespace dt

DT_EXPORT dt_status dt_layernorm_modulate_f16(dt_stream stream, int64_t M, int64_t C, const float* X, int64_t ldx,
                                              const void* scale, const void* shift, int32_t mod, float eps,
                                              uint16_t* Y, int64_t ldy) {
  using namespace dt;
  if (M < 0 || C <= 0 || mod < DT_MOD_F16 || mod > DT_MOD_AFFINE_F32) return DT_INVALID;
  if (!(eps >= 0.f) || eps - eps != 0.f) return DT_INVALID;
  if (M == 0) return DT_OK;
  if (!X || !Y || ldx < C || ldy < C) return DT_INVALID;
  if ((reinterpret_cast<uintptr_t>(X) & 3) || (reinterpret_cast<uintptr_t>(Y) & 1)) return DT_INVALID;
  const uintptr_t vec_align = mod == DT_MOD_F16 ? 1 : 3;
  if ((reinterpret_cast<uintptr_t>(scale) & vec_align) || (reinterpret_cast<uintptr_t>(shift) & vec_align)) return DT_INVALID;
  if ((M + 3) / 4 > 0x7fffffff) return DT_NO_KERNEL;
  if (const dt_status ready = device_ready(); ready != DT_OK) return ready;
  AdaLnArgs a{X, ldx, M, C, scale, shift, eps, Y, ldy};
  const bool vec = (C % 4 == 0) && (ldx % 4 == 0) && (ldy % 4 == 0) && (reinterpret_cast<uintptr_t>(X) & 15) == 0 &&
                   (reinterpret_cast<uintptr_t>(Y) & 7) == 0 &&
                   (reinterpret_cast<uintptr_t>(scale) & (mod == DT_MOD_F16 ? 7 : 15)) == 0 &&
                   (reinterpret_cast<uintptr_t>(shift) & (mod == DT_MOD_F16 ? 7 : 15)) == 0;
  if (mod == DT_MOD_F16) launch_adaln<DT_MOD_F16>(as_stream(stream), a, vec);
  else if (mod == DT_MOD_F32) launch_adaln<DT_MOD_F32>(as_stream(stream), a, vec);
  else launch_adaln<DT_MOD_AFFINE_F32>(as_stream(stream), a, vec);
  return launch_status();
}

DT_EXPORT dt_status dt_layernorm_f16(dt_stream stream, int64_t M, int64_t C, const uint16_t* X, int64_t ldx,
                                     const uint16_t* gamma, const uint16_t* beta, float eps, uint16_t* Y, int64_t ldy) {
  using namespace dt;
  if (M < 0 || C <= 0) return DT_INVALID;
  if (!(eps >= 0.f) || eps - eps != 0.f) return DT_INVALID;
  if (M == 0) return DT_OK;
  if (!X || !Y || ldx < C || ldy < C) return DT_INVALID;
  if (((reinterpret_cast<uintptr_t>(X) | reinterpret_cast<uintptr_t>(Y) | reinterpret_cast<uintptr_t>(gamma) |
        reinterpret_cast<uintptr_t>(beta)) & 1) != 0)
    return DT_INVALID;
  if ((M + 3) / 4 > 0x7fffffff) return DT_NO_KERNEL;
  if (const dt_status ready = device_ready(); ready != DT_OK) return ready;
  const LayerNorm16Args a{X, ldx, M, C, gamma, beta, eps, Y, ldy};
  const bool vec = (C % 8 == 0) && (ldx % 8 == 0) && (ldy % 8 == 0) && C <= 8 * 512 &&
                   ((reinterpret_cast<uintptr_t>(X) | reinterpret_cast<uintptr_t>(Y) | reinterpret_cast<uintptr_t>(gamma) |
                     reinterpret_cast<uintptr_t>(beta)) & 15) == 0;
  const dim3 grid((unsigned)((M + 3) / 4)), block(256);
  hipStream_t s = as_stream(stream);
  if (!vec) hipLaunchKernelGGL(layernorm16_generic_kernel, grid, block, 0, s, a);
  else if (C <= 512) hipLaunchKernelGGL((layernorm16_rows_kernel<1>), grid, block, 0, s, a);
  else if (C <= 1024) hipLaunchKernelGGL((layernorm16_rows_kernel<2>), grid, block, 0, s, a);
  else if (C <= 2048) hipLaunchKernelGGL((layernorm16_rows_kernel<4>), grid, block, 0, s, a);
  else hipLaunchKernelGGL((layernorm16_rows_kernel<8>), grid, block, 0, s, a);
  return launch_status();
}

