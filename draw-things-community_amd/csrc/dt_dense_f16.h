// K1 on plain fp16 weights with 128 x 128 tiles (128 tokens x 128 features): the weights that models ship unpacked, and the
// fp16 copies of palettized ones.
#pragma once
#include "dt_dense_kernel.h"

namespace dt {

// For launches of up to one tile per compute unit and at least five pairs of K-tiles.  512 threads = 8 waves, two per SIMD,
// each a 64 x 32 slice.  X and W go from memory straight into LDS, a pair of K-tiles (64 columns) per slot, four slots deep,
// with one barrier per pair; all of a pair's operands are read while the pair before it is multiplied (a phase of four MFMAs,
// as the kernel for all shapes has on this tile, is shorter than an LDS read takes), and reads and transfers go out between
// MFMAs: ahead of all of them they cost 1 of 10 us.
// What bounds it is the 64 bytes a clock that a compute unit takes in: 32 KB per pair, 0.25 us, where few tiles run; 0.40
// with 160 of them, which share the L2 caches' misses.  us, four slots with operands read a phase ahead / this: 40 tiles,
// K = 2048 16.2 / 13.2; 160 tiles, K = 1280 12.0 / 10.7, K = 5120 35.2 / 33.5; and the kernel for all shapes with two slots,
// two workgroups of which fit a compute unit: 32 tiles, K = 256 5.96 / 5.98, K = 128 5.27 / 5.54, K = 640 8.04 / 7.70, K =
// 2048 15.8 / 13.6.  Over 256 tiles two workgroups per compute unit are ahead (264 tiles, K = 3072 35.2 / 44.3).  (Waves
// w and w + 4 on one K-tile of each pair, 64 x 64 slices: eight operand reads per pair instead of twelve, but the sums then
// meet in LDS behind the loop: K = 1280 10.8, K = 2048 13.2, K = 256 6.5.)
template <bool POST, bool LORA>
__global__ void __launch_bounds__(512, 2) dense_f16_kernel(const DenseArgs a) {
  constexpr int BM = 128, BN = 128;
  constexpr int NS = 4;                     // slots
  constexpr int PROW = 2 * BK;              // halfs per row of a slot
  constexpr int PARTS = BM * (BK / 4) / 512;  // 16-byte chunks of X, and of W, per thread per pair
  constexpr int TILE_B = BM * PROW * 2;     // bytes of one operand of a slot
  constexpr int SLOT_B = 2 * TILE_B;
  static_assert(NS % 2 == 0 && (NS - 1) * 2 * PARTS < 16, "slots");
  __shared__ __attribute__((aligned(4096))) unsigned char smem[NS * SLOT_B];  // (the epilogue parks the tile's 32 KB here)

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wn = wave & 1, wm = ((wave >> 1) & 1) | ((wave >> 2) << 1);

  const TileAt at = tile_at(a, xcd_order(blockIdx.x, a.total_tiles));
  const DenseGroup g = a.g[at.group];
  const DenseWeight w = a.w[at.weight];
  const int n0 = (at.tn - w.tile_begin) * BN;
  const int m0 = at.tm * BM;
  const int K = a.k;
  const int n_pairs = K / (2 * BK);

  // a transfer fills 1 KB of a slot = 8 rows; see dense_qx_kernel
  uint32_t x_off[PARTS], w_off[PARTS];
#pragma unroll
  for (int i = 0; i < PARTS; i++) {
    const int row = 8 * (wave * PARTS + i) + (lane >> 3);
    const int c8 = pair_chunk(row, lane & 7);
    int gm = m0 + row, gn = n0 + row;
    if (gm >= g.m) gm = g.m - 1;
    if (gn >= w.n) gn = w.n - 1;
    x_off[i] = (uint32_t)(((int64_t)gm * g.ldx + c8 * 8) * 2);
    w_off[i] = (uint32_t)(((int64_t)gn * K + c8 * 8) * 2);
  }
  const char* const xbase = reinterpret_cast<const char*>(g.x);
  const char* const wbase = reinterpret_cast<const char*>(w.data);
  // part p of the transfer of pair q into a slot (pairs past the end re-read the last one, harmlessly)
  auto issue_part = [&](int slot, int q, int p) __attribute__((always_inline)) {
    if (q >= n_pairs) q = n_pairs - 1;
    const int64_t kb = (int64_t)q * (4 * BK);
    const int i = p >> 1;
    const uint32_t dst = lds_address(smem) + (uint32_t)(slot * SLOT_B + (p & 1) * TILE_B + (wave * PARTS + i) * 1024);
    if (p & 1) load_to_lds_16(wbase + kb, w_off[i], dst);
    else load_to_lds_16(xbase + kb, x_off[i], dst);
  };

  // v_mfma_f32_16x16x32_f16: A operand = W rows, B operand = X rows; lane holds row (lane & 15), k 8 * (lane / 16) .. + 7
  const int l16 = lane & 15, quad = lane >> 4;
  const int xrow = wm * 32 + l16, wrow = wn * 64 + l16;  // rows 16 apart share a swizzle; the K-tile of the pair is xor'ed
  const int x_lane = xrow * PROW + (pair_chunk(xrow, quad) << 3), w_lane = wrow * PROW + (pair_chunk(wrow, quad) << 3);
  half8_t fx[2][2][2], fw[2][2][4];  // [set][K-tile][block]
  // operand r of the twelve of a pair
  auto read_part = [&](int set, int slot, int r) __attribute__((always_inline)) {
    const int par = r / 6, i = r % 6;
    const half_t* const xs = reinterpret_cast<const half_t*>(smem + slot * SLOT_B) + (x_lane ^ (32 * par));
    const half_t* const ws = reinterpret_cast<const half_t*>(smem + slot * SLOT_B + TILE_B) + (w_lane ^ (32 * par));
    if (i < 4) fw[set][par][i] = *reinterpret_cast<const half8_t*>(ws + i * 16 * PROW);
    else fx[set][par][i - 4] = *reinterpret_cast<const half8_t*>(xs + (i - 4) * 16 * PROW);
  };
  float4_t acc[4][2];
#pragma unroll
  for (int i = 0; i < 4; i++)
#pragma unroll
    for (int j = 0; j < 2; j++) acc[i][j] = float4_t{0.f, 0.f, 0.f, 0.f};

#pragma unroll
  for (int s = 0; s < NS; s++)
#pragma unroll
    for (int p = 0; p < 2 * PARTS; p++) issue_part(s, s, p);
  __builtin_amdgcn_s_waitcnt(kWaitVm0Lgkm0 | (NS - 1) * 2 * PARTS);  // pair 0
  __syncthreads();
#pragma unroll
  for (int r = 0; r < 12; r++) read_part(0, 0, r);

  // Pair q, whose operands are in set q % 2 and were read from slot q % NS: that slot is free once every wave's reads are back.
  auto pair = [&](int q, int set, int slot) __attribute__((always_inline)) {
    __builtin_amdgcn_s_waitcnt(kWaitVm0Lgkm0 | (NS - 2) * 2 * PARTS);  // pair q + 1 has landed, pair q is in registers
    __syncthreads();
#pragma unroll
    for (int m = 0; m < 16; m++) {
      __builtin_amdgcn_sched_barrier(0);
      const int par = m >> 3, i = m & 3, j = (m >> 2) & 1;
      acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(fw[set][par][i], fx[set][par][j], acc[i][j], 0, 0, 0);
      __builtin_amdgcn_sched_barrier(0);
      if (m < 6) {
        read_part(set ^ 1, slot + 1 < NS ? slot + 1 : 0, 2 * m);
        read_part(set ^ 1, slot + 1 < NS ? slot + 1 : 0, 2 * m + 1);
      } else if (m < 6 + 2 * PARTS) {
        issue_part(slot, q + NS, m - 6);
      }
    }
    __builtin_amdgcn_sched_barrier(0);
  };
  // rounds of NS pairs, so that slots and register sets are constants
  int q = 0;
  for (; q + NS <= n_pairs; q += NS) {
#pragma unroll
    for (int i = 0; i < NS; i++) pair(q + i, i & 1, i);
  }
#pragma unroll
  for (int i = 0; i < NS - 1; i++)
    if (q + i < n_pairs) pair(q + i, i & 1, i);

  __builtin_amdgcn_s_waitcnt(kWaitVm0Lgkm0);  // nothing is in flight into LDS any more
  __syncthreads();
  dense_epilogue<64, 32, POST, LORA>(acc, smem, wave, lane, n0 + wn * 64, (int64_t)m0 + wm * 32, w, g.m, a.lora);
}

}  // namespace dt
