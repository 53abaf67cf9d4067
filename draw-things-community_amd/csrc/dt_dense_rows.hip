// K1r: Dense with few rows (a conditioning vector, a short prompt): Y = X W^T where reading W is the work.
//
// What bounds it: the bytes of the packed weight and, behind them, the lookups (one LDS gather per 64 weights).  So every
// wave streams whole index granules of its own 16 weight rows straight from memory into registers -- nothing of W goes
// through LDS but the palettes -- looks them up, and uses the result as the A operand of v_mfma_f32_16x16x32_f16 with
// the rows of X as columns.  A wave keeps 16 * RB features; the waves of a workgroup take turns at stretches of
// 128 k, so that they read consecutive memory, and add their sums up in LDS at the end.
// 1 x 3072 -> 6 x 3072 q8p: 17.1 us, 3.4 TB/s of its 58 MB (128 x 128 tiles: 66 us, 0.87 TB/s); plain fp16 5120 ->
// 6 x 5120: 52 us, 6.0 TB/s (78 us).
#include "dt_dense_launch.h"
#include "dt_dense_rows.h"

namespace dt {

typedef uint32_t u32x4_a4 __attribute__((ext_vector_type(4), aligned(4)));

constexpr int kRowsPalBytes = 32768;

// TM: token blocks of 16; RB: feature blocks of 16; NW: waves
template <int Q, int TM, int RB, int NW>
__global__ void __launch_bounds__(64 * NW) dense_rows_kernel(const DenseArgs a) {
  constexpr int FB = 16 * RB;
  constexpr int ND = Q == 16 ? 16 : Q;  // dwords of 32 weights or indices
  constexpr int RED_BYTES = NW * TM * 16 * (FB + 1) * 4;
  constexpr int PAL_BYTES = Q == 16 ? 16 : kRowsPalBytes;
  __shared__ __attribute__((aligned(16))) unsigned char smem[RED_BYTES > PAL_BYTES ? RED_BYTES : PAL_BYTES];
  uint16_t* const pal = reinterpret_cast<uint16_t*>(smem);
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int l16 = lane & 15, c = lane >> 4;
  int wi = 0;
#pragma unroll
  for (int i = 1; i < kMaxWeights; i++)
    if (i < a.g[0].w_end && (int)blockIdx.x >= a.w[i].tile_begin) wi = i;
  const DenseWeight w = a.w[wi];
  const int n0 = ((int)blockIdx.x - w.tile_begin) * FB;
  const int K = a.k, M = a.g[0].m;
  const int n_gran = K / 32, n_step = (n_gran + 3) / 4;
  const QxLayout lay = make_layout(Q == 16 ? 8 : Q, a.nib);
  const uint32_t nib = (uint32_t)a.nib;

  // this lane's cursors: granule 4 * step + c of each of its rows
  uint32_t raw[2][RB][ND];
  int64_t blk[RB];
  uint32_t pos[RB];
  int32_t slot[2][RB];
  int64_t row_e[RB];
  int64_t blk0 = 0;
  if constexpr (Q != 16) blk0 = (int64_t)n0 * K / a.nib;
#pragma unroll
  for (int b = 0; b < RB; b++) {
    const int gn = n0 + 16 * b + l16 < w.n ? n0 + 16 * b + l16 : w.n - 1;
    row_e[b] = (int64_t)gn * K;
    if constexpr (Q != 16) {
      const int64_t e = row_e[b] + 32 * (4 * wave + c);
      blk[b] = e / a.nib;
      pos[b] = (uint32_t)(e - blk[b] * a.nib);
    }
  }
  auto fetch_w = [&](int buf, int step) {
    const bool on = 4 * step + c < n_gran;  // (a lane past the row's end reads its first granule)
#pragma unroll
    for (int b = 0; b < RB; b++) {
      const uint32_t* src;
      if constexpr (Q == 16) {
        src = reinterpret_cast<const uint32_t*>(w.data) + (row_e[b] + (on ? 32 * (4 * step + c) : 0)) / 2;
      } else {
        const int64_t bb = on ? blk[b] : blk0;
        src = reinterpret_cast<const uint32_t*>(w.data + index_byte_offset(lay, bb, on ? pos[b] : 0));
        slot[buf][b] = (int32_t)(bb - blk0);
        pos[b] += 128 * NW;
        if (pos[b] >= nib) {
          const uint32_t q = pos[b] / nib;
          blk[b] += q;
          pos[b] -= q * nib;
        }
      }
#pragma unroll
      for (int i = 0; i + 4 <= ND; i += 4) {
        const u32x4_a4 v = *reinterpret_cast<const u32x4_a4*>(src + i);
#pragma unroll
        for (int e = 0; e < 4; e++) raw[buf][b][i + e] = v[e];
      }
#pragma unroll
      for (int i = ND / 4 * 4; i < ND; i++) raw[buf][b][i] = src[i];
    }
  };
  const uint16_t* xrow[TM];
#pragma unroll
  for (int t = 0; t < TM; t++) {
    const int m = 16 * t + l16 < M ? 16 * t + l16 : M - 1;
    xrow[t] = a.g[0].x + (int64_t)m * a.g[0].ldx + 32 * c;
  }

  float4_t acc[TM][RB];
#pragma unroll
  for (int t = 0; t < TM; t++)
#pragma unroll
    for (int b = 0; b < RB; b++) acc[t][b] = float4_t{0.f, 0.f, 0.f, 0.f};

  if (wave < n_step) fetch_w(0, wave);
  if constexpr (Q != 16) {
    const int last_row = n0 + FB <= w.n ? n0 + FB - 1 : w.n - 1;
    const int n_pal = (int)(((int64_t)last_row * K + K - 1) / a.nib - blk0 + 1);
    for (int i = tid; i < n_pal << (Q - 1); i += 64 * NW)
      reinterpret_cast<uint32_t*>(pal)[i] =
          reinterpret_cast<const uint32_t*>(w.data + palette_offset(lay, blk0 + (i >> (Q - 1))))[i & ((1 << (Q - 1)) - 1)];
    __syncthreads();
  }
  auto step_once = [&](int buf, int step) {
    uint4_t x[TM][4];
    const bool on = 4 * step + c < n_gran;
#pragma unroll
    for (int t = 0; t < TM; t++)
#pragma unroll
      for (int j = 0; j < 4; j++) x[t][j] = *reinterpret_cast<const uint4_t*>(xrow[t] + (on ? 128 * step : -32 * c) + 8 * j);
    if (step + NW < n_step) fetch_w(buf ^ 1, step + NW);
    if (4 * step + 3 >= n_gran) {  // uniform: the row ends inside this stretch
#pragma unroll
      for (int t = 0; t < TM; t++)
#pragma unroll
        for (int j = 0; j < 4; j++) x[t][j] = on ? x[t][j] : uint4_t{0, 0, 0, 0};
    }
#pragma unroll
    for (int b = 0; b < RB; b++) {
      uint32_t pk[16];  // the granule as fp16 pairs
      if constexpr (Q == 16) {
#pragma unroll
        for (int i = 0; i < 16; i++) pk[i] = raw[buf][b][i];
      } else {
        uint32_t idx[32];
        unpack32<Q>(raw[buf][b], idx);
        const uint16_t* mine = pal + (slot[buf][b] << Q);
#pragma unroll
        for (int i = 0; i < 16; i++) pk[i] = (uint32_t)mine[idx[2 * i]] | ((uint32_t)mine[idx[2 * i + 1]] << 16);
      }
      if (4 * step + 3 >= n_gran) {
#pragma unroll
        for (int i = 0; i < 16; i++) pk[i] = on ? pk[i] : 0;
      }
#pragma unroll
      for (int j = 0; j < 4; j++) {
        const half8_t wf = __builtin_bit_cast(half8_t, uint4_t{pk[4 * j], pk[4 * j + 1], pk[4 * j + 2], pk[4 * j + 3]});
#pragma unroll
        for (int t = 0; t < TM; t++)
          acc[t][b] = __builtin_amdgcn_mfma_f32_16x16x32_f16(wf, __builtin_bit_cast(half8_t, x[t][j]), acc[t][b], 0, 0, 0);
      }
    }
  };
  for (int step = wave; step < n_step; step += 2 * NW) {
    step_once(0, step);
    if (step + NW < n_step) step_once(1, step + NW);
  }
  __syncthreads();  // the palettes' LDS is free

  // sums as [wave][token][feature]: lane holds token l16 and features 4 c .. 4 c + 3 of each block
  float* red = reinterpret_cast<float*>(smem);
#pragma unroll
  for (int t = 0; t < TM; t++)
#pragma unroll
    for (int b = 0; b < RB; b++)
#pragma unroll
      for (int v = 0; v < 4; v++) red[((wave * TM + t) * 16 + l16) * (FB + 1) + 16 * b + 4 * c + v] = acc[t][b][v];
  __syncthreads();
  for (int i = tid; i < TM * 16 * FB; i += 64 * NW) {
    const int t = i / FB, f = i % FB;
    const int64_t ni = n0 + f;
    if (t >= M || ni >= w.n) continue;
    float s = 0.f;
#pragma unroll
    for (int p = 0; p < NW; p++) s += red[(p * TM * 16 + t) * (FB + 1) + f];
    if (w.bias) s += (float)bits_to_half(w.bias[ni]);
    store_post(w, t, ni, round_f16(s));
  }
}

template <int Q, int TM>
static void launch_rows(hipStream_t s, const DenseArgs& a, int rb, int nw) {
  const dim3 grid((unsigned)a.total_tiles);
  if (nw == 4) {
    if (rb == 2) hipLaunchKernelGGL((dense_rows_kernel<Q, TM, 2, 4>), grid, dim3(256), 0, s, a);
    else hipLaunchKernelGGL((dense_rows_kernel<Q, TM, 1, 4>), grid, dim3(256), 0, s, a);
  } else {
    if (rb == 2) hipLaunchKernelGGL((dense_rows_kernel<Q, TM, 2, 8>), grid, dim3(512), 0, s, a);
    else hipLaunchKernelGGL((dense_rows_kernel<Q, TM, 1, 8>), grid, dim3(512), 0, s, a);
  }
}

template <int Q>
static dt_status launch_rows_q(hipStream_t s, const DenseArgs& a, int rb) {
  // Eight waves share a block's K while there are fewer than three blocks per compute unit; beyond, four, so that more
  // blocks are in flight at once (3072 -> 6 x 3072 q8p, one row: 17.1 us against 18.0; 3072 -> 3072: 6.3 / 5.6).
  const int nw = a.total_tiles >= 768 ? 4 : 8;
  if (a.g[0].m <= 16) launch_rows<Q, 1>(s, a, rb, nw);
  else if (a.g[0].m <= 32) launch_rows<Q, 2>(s, a, rb, nw);
  else launch_rows<Q, 4>(s, a, rb, nw);
  return launch_status();
}

int dense_rows_features(int64_t M, int64_t K, int qbits, int nib, int64_t n_total) {
  // Up to where the 128-wide tiles catch up.  They read a packed weight no faster at 64 rows than at one (us, 3072 ->
  // 6 x 3072 q8p: 66-70 against 17 at 1 row, 29 at 32, 49 at 64); with plain fp16 weights, which cost them no
  // unpacking, they do once they have enough features to fill the chip (3072 -> 6 x 3072: 32 against 20 at 1 row, 27 at
  // 16, 37 at 32; 5120 -> 5120: 48 against 32 at 64 rows).
  if (M > kRowsMax || (qbits == 16 && M > 16 && n_total > 8192)) return 0;
  // Blocks of 32 features read X half as often, which pays from the second token block on if the launch still fills the
  // chip (5120 -> 5120 q8p at 32 rows: 18.5 us against 25.2, at one row 12.7 against 12.1; 3072 -> 3072 at 32: 12.2 / 9.5).
  int fb = M > 16 && n_total >= 5120 ? 32 : 16;
  if (qbits != 16) {
    const auto fits = [&](int f) { return (f * K / nib + 2) * ((int64_t)2 << qbits) <= kRowsPalBytes; };
    if (!fits(fb)) fb = 16;
    if (!fits(fb)) return 0;
  }
  return fb;
}

dt_status dense_rows_launch(hipStream_t s, const DenseArgs& a, int qbits, int features) {
  const int rb = features / 16;
  switch (qbits) {
    case 4: return launch_rows_q<4>(s, a, rb);
    case 5: return launch_rows_q<5>(s, a, rb);
    case 6: return launch_rows_q<6>(s, a, rb);
    case 7: return launch_rows_q<7>(s, a, rb);
    case 8: return launch_rows_q<8>(s, a, rb);
    case 16: return launch_rows_q<16>(s, a, rb);
  }
  return DT_INVALID;
}

}  // namespace dt
