// K1a: Dense for the shapes the tiled kernel (dt_dense_kernel.h) does not take -- K no multiple of 64, blocks that are
// no multiple of 32, rows or weights off the 16-byte grid -- on the matrix instruction all the same.
//
// What bounds it: the launches are small (odd widths come with small layers), so it is latency: of the index and X
// loads, hidden by fetching a K-tile ahead into registers, of the unpacking of a tile's indices, and of the K loop, kept short by
// giving the four waves of a small tile a quarter of every K-tile each and, where compute units have a workgroup to themselves, by
// groups of four waves that take every second or fourth K-tile (their sums meet in LDS).  231 x 1000 -> 1001 q8p: 8.6 us (13.3 with one
// group, 10.1 with two; 6.8 / 8.6 / 7.4 with plain fp16 weights), where one thread per output, walking K on its own, took 1105.
// (One group that fetches two to four K-tiles ahead changes nothing: 13.0 - 13.2 us.)
#include "dt_dense_any.h"

#include "dt_dense_kernel.h"
#include "dt_layout.h"

namespace dt {

// (the part reads words at any address, one instruction each)
typedef uint32_t u32_any __attribute__((aligned(1)));
typedef uint16_t u16_any __attribute__((aligned(1)));
typedef uint32_t u32x4_any __attribute__((ext_vector_type(4), aligned(2)));

// 16 halfs of a row; with CUT those from `left` on are zero and not read.  (Two forms because a lane's partial load
// would make every other lane wait for its whole one: they write the same registers.)
template <bool CUT>
__device__ __forceinline__ void load_halfs16(const uint16_t* p, int left, uint32_t (&raw)[8]) {
  if constexpr (!CUT) {
#pragma unroll
    for (int c = 0; c < 2; c++) {
      const u32x4_any v = *reinterpret_cast<const u32x4_any*>(p + 8 * c);
#pragma unroll
      for (int i = 0; i < 4; i++) raw[4 * c + i] = v[i];
    }
  } else {
    uint32_t h[16];
#pragma unroll
    for (int i = 0; i < 16; i++) h[i] = p[i < left ? i : 0];
#pragma unroll
    for (int i = 0; i < 8; i++)
      raw[i] = (2 * i < left ? h[2 * i] : 0) | (2 * i + 1 < left ? h[2 * i + 1] << 16 : 0);
  }
}

// BT x BT outputs per 256-thread workgroup (BT = 64: 2 x 2 waves of 32 x 32; BT = 32: every wave computes the whole
// tile over its own quarter of each K-tile).  A K-tile is 4096 / BT wide, so that a thread always stages 16 consecutive
// k of one X row and of one weight row.
// G groups of 256 threads take every G-th K-tile each, and their sums meet in LDS.
template <int Q, int BT, int G>
__global__ void __launch_bounds__(256 * G) dense_any_kernel(const DenseAnyArgs a) {
  constexpr int BKA = 4096 / BT, RUNS = BKA / 16;
  constexpr int LDR = BKA + 8;                 // halfs per LDS row: 16 consecutive rows start on 16 different bank groups
  constexpr int BUF = BT * LDR;                // halfs per operand and stage
  constexpr int HW = Q == 16 ? 8 : (Q + 1) / 2;  // dwords that hold a thread's 16 weights or indices
  constexpr int NRAW = Q == 16 ? 8 : HW + 1;     // ... at any byte offset
  constexpr int OUT_LD = BT + 1;
  constexpr int PARTS = (BT == 32 ? 4 : 1) * G;  // sums of every output
  static_assert(PARTS * BT * OUT_LD * 4 <= G * 4 * BUF * 2, "the output tile reuses the operand buffers");
  __shared__ __attribute__((aligned(16))) half_t all_tiles[G * 4 * BUF];
  __shared__ __attribute__((aligned(4))) uint16_t pal_lds[Q == 16 ? 2 : kAnyPalBytes / 2];

  const int tid = G == 1 ? threadIdx.x : threadIdx.x & 255, lane = tid & 63, wave = tid >> 6;
  const int group = G == 1 ? 0 : __builtin_amdgcn_readfirstlane(threadIdx.x >> 8);
  half_t* const tiles = all_tiles + group * 4 * BUF;
  const int l32 = lane & 31, hi = lane >> 5;
  const int64_t m0 = (blockIdx.x % a.tiles_m) * BT, n0 = (blockIdx.x / a.tiles_m) * BT;
  const int row = tid / RUNS, run = tid % RUNS;
  const int64_t gm = m0 + row, gn = any_row(n0 + row, a.n);
  const uint16_t* xr = a.x + (gm < a.m ? gm : 0) * a.ldx;
  const QxLayout lay = make_layout(Q == 16 ? 8 : Q, Q == 16 ? 32 : a.nib);
  const int nib = lay.nib;

  // the output feature that this thread finishes (in several rows), and its bias
  const int of = threadIdx.x % BT;
  const float bias = a.bias && n0 + of < a.n ? (float)bits_to_half(a.bias[n0 + of]) : 0.f;

  // palettes of every block the tile's rows touch, asked for four dwords at a time: one trip to memory, not one for each
  // (us, q8p, one by one / four at a time, the bias likewise ahead: 231 x 1000 -> 1001 13.3 / 13.1, 1000 rows 25.2 / 24.1, 700 x 300 ->
  // 2200 17.0 / 16.1)
  int64_t blk0 = 0;
  if constexpr (Q != 16) {
    if (a.pal_shared) {
      const AnyBlocks held = any_blocks(n0, BT, a.n, a.k, nib);
      blk0 = held.first;
      const int n_pal = held.count << (Q - 1);
      for (int i0 = threadIdx.x; i0 < n_pal; i0 += 4 * 256 * G) {
        uint32_t v[4];
#pragma unroll
        for (int j = 0; j < 4; j++) {
          const int i = i0 + 256 * G * j < n_pal ? i0 + 256 * G * j : i0;
          v[j] = reinterpret_cast<const u32_any*>(a.w + palette_offset(lay, blk0 + (i >> (Q - 1))))[i & ((1 << (Q - 1)) - 1)];
        }
#pragma unroll
        for (int j = 0; j < 4; j++)
          if (i0 + 256 * G * j < n_pal) reinterpret_cast<uint32_t*>(pal_lds)[i0 + 256 * G * j] = v[j];
      }
    }
  }

  const bool runs_ok = any_by_words(NRAW, a.w_bytes, nib);  // (otherwise index by index)
  AnyCursor next = {0, 0};  // this thread's next weight run
  if constexpr (Q != 16) next = any_cursor(gn, a.k, group * BKA + run * 16, nib);

  // NRAW dwords from byte p of the packed buffer on; the result is the number of bytes by which they are early.
  auto load_raw = [&](int64_t p, uint32_t (&raw)[NRAW]) {
    const int64_t q = any_words_at(p, NRAW, a.w_bytes);
    const u32_any* src = reinterpret_cast<const u32_any*>(a.w + q);
#pragma unroll
    for (int i = 0; i < NRAW; i++) raw[i] = src[i];
    return (int)(p - q);
  };
  auto drop_bytes = [&](uint32_t (&raw)[NRAW], int n) {
    if (n <= 0) return;
    for (; n >= 4; n -= 4) {
#pragma unroll
      for (int i = 0; i + 1 < NRAW; i++) raw[i] = raw[i + 1];
    }
#pragma unroll
    for (int i = 0; i < NRAW; i++)
      raw[i] = (uint32_t)((((uint64_t)(i + 1 < NRAW ? raw[i + 1] : 0) << 32) | raw[i]) >> (8 * n));
  };
  // ... as the big-endian bit string that starts `sh` (0 .. 7) bits in
  auto bit_string = [&](const uint32_t (&raw)[NRAW], int sh, uint32_t (&be)[HW + 1]) {
    if constexpr (Q != 16) {
#pragma unroll
      for (int i = 0; i < HW; i++) {
        const uint64_t two = ((uint64_t)__builtin_bswap32(raw[i]) << 32) | __builtin_bswap32(raw[i + 1]);
        be[i] = (uint32_t)(two >> (32 - sh));
      }
      be[HW] = 0;
    }
  };

  uint32_t xraw[8], wraw[NRAW], wraw2[NRAW];
  int w_left = 0;  // weights of the fetched run that exist
  int w_head = 0;  // ... of which this many lie in its first block, the others in the next one
  int early = 0, early2 = 0, sh2 = 0;
  bool two = false;  // some lane's run crosses into another block
  AnyCursor cur = {0, 0};
  auto fetch = [&](int kt) {
    const int64_t k0 = (int64_t)kt * BKA + run * 16;
    w_left = any_run(k0, a.k);
    const bool whole = (int64_t)(kt + 1) * BKA <= a.k;  // uniform
    if (whole) load_halfs16<false>(xr + k0, 16, xraw);
    else load_halfs16<true>(xr + (w_left ? k0 : 0), w_left, xraw);
    if constexpr (Q == 16) {
      const uint16_t* wr = reinterpret_cast<const uint16_t*>(a.w) + gn * a.k;
      if (whole) load_halfs16<false>(wr + k0, 16, wraw);
      else load_halfs16<true>(wr + (w_left ? k0 : 0), w_left, wraw);
    } else {
      cur = next;
      w_head = any_run_head(cur, w_left, nib);
      if (runs_ok) {
        early = load_raw(index_byte_offset(lay, w_left ? cur.blk : 0, w_left ? cur.r : 0), wraw);
        two = __builtin_amdgcn_ballot_w64(w_head < w_left) != 0;
        if (two) {
          const int64_t bit = w_head < w_left ? any_rest_bit(lay, cur, w_head) : 0;
          sh2 = (int)(bit & 7);
          early2 = load_raw(bit >> 3, wraw2);
        }
      }
      any_advance(next, G * BKA, nib);
    }
  };
  auto stage = [&](int buf) {
    half_t* xs = tiles + buf * 2 * BUF + row * LDR + run * 16;
    half_t* ws = xs + BUF;
    *reinterpret_cast<uint4_t*>(xs) = uint4_t{xraw[0], xraw[1], xraw[2], xraw[3]};
    *reinterpret_cast<uint4_t*>(xs + 8) = uint4_t{xraw[4], xraw[5], xraw[6], xraw[7]};
    if constexpr (Q == 16) {
      *reinterpret_cast<uint4_t*>(ws) = uint4_t{wraw[0], wraw[1], wraw[2], wraw[3]};
      *reinterpret_cast<uint4_t*>(ws + 8) = uint4_t{wraw[4], wraw[5], wraw[6], wraw[7]};
    } else {
      uint32_t v[16];
#pragma unroll
      for (int j = 0; j < 16; j++) v[j] = 0;
      // weights [from, to) of the run from the palette of block b
      auto look_up = [&](const uint32_t (&raw)[NRAW], int sh, int64_t b, int from, int to) {
        uint32_t be[HW + 1];
        bit_string(raw, sh, be);
        uint32_t got[16];
        if (a.pal_shared) {  // uniform
          const uint16_t* lp = pal_lds + ((int)(b - blk0) << Q);
#pragma unroll
          for (int j = 0; j < 16; j++) got[j] = lp[own_index<Q, HW>(be, j)];
        } else {
          const u16_any* gp = reinterpret_cast<const u16_any*>(a.w + palette_offset(lay, b));
#pragma unroll
          for (int j = 0; j < 16; j++) got[j] = gp[own_index<Q, HW>(be, j)];
        }
#pragma unroll
        for (int j = 0; j < 16; j++) v[j] = j >= from && j < to ? got[j] : v[j];
      };
      if (runs_ok) {
        drop_bytes(wraw, early);
        look_up(wraw, (int)((cur.r * Q) & 7), w_left ? cur.blk : blk0, 0, w_head);
        if (two) {
          drop_bytes(wraw2, early2);
          look_up(wraw2, sh2, w_head < w_left ? cur.blk + 1 : blk0, w_head, w_left);
        }
      } else {
        int64_t b = cur.blk;
        uint32_t rr = cur.r;
#pragma unroll
        for (int j = 0; j < 16; j++)
          if (j < w_left) {
            const uint8_t* base = a.w + palette_offset(lay, b);
            v[j] = reinterpret_cast<const u16_any*>(base)[load_index(base + lay.pal_bytes, rr, Q)];
            if (++rr == (uint32_t)nib) {
              rr = 0;
              b++;
            }
          }
      }
#pragma unroll
      for (int h = 0; h < 2; h++)
        *reinterpret_cast<uint4_t*>(ws + 8 * h) =
            uint4_t{v[8 * h] | (v[8 * h + 1] << 16), v[8 * h + 2] | (v[8 * h + 3] << 16),
                    v[8 * h + 4] | (v[8 * h + 5] << 16), v[8 * h + 6] | (v[8 * h + 7] << 16)};
    }
  };

  float16_t acc;
#pragma unroll
  for (int v = 0; v < 16; v++) acc[v] = 0.f;
  const int wn = BT == 64 ? wave & 1 : 0, wm = BT == 64 ? wave >> 1 : 0;
  const int ks0 = BT == 64 ? 0 : 2 * wave;
  constexpr int NKS = BT == 64 ? 4 : 2;
  const int nkt = (int)((a.k + BKA - 1) / BKA), rounds = (nkt + G - 1) / G;  // (a K-tile past the end is zeros)
  fetch(group);
  __syncthreads();  // palettes visible
  stage(0);
  __syncthreads();
  for (int kt = 0; kt < rounds; kt++) {
    const bool more = kt + 1 < rounds;
    if (more) fetch((kt + 1) * G + group);
    const half_t* xs = tiles + (kt & 1) * 2 * BUF + (wm * 32 + l32) * LDR + 8 * hi;
    const half_t* ws = tiles + (kt & 1) * 2 * BUF + BUF + (wn * 32 + l32) * LDR + 8 * hi;
#pragma unroll
    for (int s = 0; s < NKS; s++)
      acc = __builtin_amdgcn_mfma_f32_32x32x16_f16(*reinterpret_cast<const half8_t*>(ws + 16 * (ks0 + s)),
                                                   *reinterpret_cast<const half8_t*>(xs + 16 * (ks0 + s)), acc, 0, 0, 0);
    if (more) stage((kt + 1) & 1);
    __syncthreads();
  }

  // Sums to LDS as [token][feature], then element by element with consecutive features in consecutive lanes.
  float* outs = reinterpret_cast<float*>(all_tiles) + (BT == 32 ? group * 4 + wave : group) * BT * OUT_LD;
#pragma unroll
  for (int v = 0; v < 16; v++)
    outs[(wm * 32 + l32) * OUT_LD + wn * 32 + 8 * (v >> 2) + 4 * hi + (v & 3)] = acc[v];
  __syncthreads();
  const float* sums = reinterpret_cast<const float*>(all_tiles);
  for (int t = threadIdx.x / BT; t < BT; t += 256 * G / BT) {
    const int64_t mi = m0 + t, ni = n0 + of;
    if (mi >= a.m || ni >= a.n) continue;
    float s = sums[t * OUT_LD + of];
    if constexpr (PARTS > 1) {
#pragma unroll
      for (int p = 1; p < PARTS; p++) s += sums[(p * BT + t) * OUT_LD + of];
    }
    if (a.bias) s += bias;
    store_post(a, mi, ni, round_f16(s));
  }
}

template <int Q>
static void launch_any(hipStream_t s, const DenseAnyArgs& a, bool big, int groups, unsigned grid) {
  const dim3 block(256 * (unsigned)groups);
  if (big) {
    if (groups == 4) hipLaunchKernelGGL((dense_any_kernel<Q, 64, 4>), dim3(grid), block, 0, s, a);
    else hipLaunchKernelGGL((dense_any_kernel<Q, 64, 1>), dim3(grid), block, 0, s, a);
  } else {
    if (groups == 4) hipLaunchKernelGGL((dense_any_kernel<Q, 32, 4>), dim3(grid), block, 0, s, a);
    else if (groups == 2) hipLaunchKernelGGL((dense_any_kernel<Q, 32, 2>), dim3(grid), block, 0, s, a);
    else hipLaunchKernelGGL((dense_any_kernel<Q, 32, 1>), dim3(grid), block, 0, s, a);
  }
}

dt_status dense_any_launch(hipStream_t s, DenseAnyArgs a) {
  if (a.m <= 0 || a.n <= 0) return DT_OK;
  const auto tiles = [&](int t) { return ((a.m + t - 1) / t) * ((a.n + t - 1) / t); };
  // The 64 x 64 tile halves what is read and unpacked per output but takes twice as long for a K-tile pair; with one group of waves it
  // wins once there are more of them than compute units.  Up to there groups share K out: as many as K is long enough for where 32 x 32
  // tiles have a compute unit each, and on 64 x 64 tiles where there are more of the small ones.  us, q8p (fp16):
  //   small tiles, 1 / 2 / 4 groups: 231 x 1000 -> 1001 13.3 / 10.1 / 8.6 (8.6 / 7.4 / 6.8), 130 x 700 -> 500 11.2 / 8.9 / 8.8 (7.7 / 6.7 / 7.3), 1 x 2555 ->
  //     2555 23.6 / 17.3 / 15.0 (13.3 / 10.8 / 9.8), 70 x 100 -> 96 5.6 / 5.7 / 6.3; where they share compute units 500 x 1000 -> 1001 15.4 / 18.1 / 15.4
  //   small ones / 64 wide, 1 / 4 groups: 500 x 1000 -> 1001 15.4 / 24.6 / 13.4 (10.3 / 15.4 / 9.9), 1000 rows 26.9 / 24.9 / 13.7 (15.9 / 15.8 / 10.4), 100
  //     x 300 -> 2200 9.1 / 13.7 / 10.2, 333 x 90 -> 1500 7.7 / 10.8 / 8.1; over 256 of them 1000 x 2500 -> 2500 112 / 70.6 / 73.9, 700 x 300 -> 2200 19.3
  //     / 16.3 / 18.9
  //   ... and up to two of the small ones for a compute unit one or two groups on these hold their own: on plain weights against the wide ones, which
  //     wait for memory (702 x 2452 -> 476 15.3 with two / 24.4, 265 x 2141 -> 1494 19.5 / 24.6, 240 x 1474 -> 1595 14.3 / 12.3; up to 1152 inputs with one, 233 x 547 ->
  //     2006 9.8 / 11.5), and otherwise where the wide ones' last round of K-tiles is short (159 x 1052 -> 1650 15.0 with one / 16.5, 1000 inputs 13.8 / 13.6)
  const int64_t small_tiles = tiles(32), k_tiles = (a.k + 127) / 128, wide_rounds = ((a.k + 63) / 64 + 3) / 4;
  const bool two_each = small_tiles > 256 && small_tiles <= 512, plain = a.qbits == 16;
  const bool shared_out = tiles(64) <= 256 && small_tiles > 256 && a.k > 512 && !(two_each && (plain || 20 * k_tiles <= 37 * wide_rounds));
  const bool big = shared_out || tiles(64) >= 256;
  const int groups = shared_out ? 4 : big || k_tiles < 2 ? 1 : small_tiles > 256 ? (two_each && plain && a.k > 1152 ? 2 : 1) : k_tiles >= (plain ? 8 : 6) ? 4 : 2;
  const int BT = big ? 64 : 32;
  const int64_t grid = tiles(BT);
  if (grid > 0x7fffffff) return DT_NO_KERNEL;
  a.tiles_m = (a.m + BT - 1) / BT;
  a.pal_shared = a.qbits != 16 && any_pal_shared(BT, a.k, a.qbits, a.nib);
  switch (a.qbits) {
    case 4: launch_any<4>(s, a, big, groups, (unsigned)grid); break;
    case 5: launch_any<5>(s, a, big, groups, (unsigned)grid); break;
    case 6: launch_any<6>(s, a, big, groups, (unsigned)grid); break;
    case 7: launch_any<7>(s, a, big, groups, (unsigned)grid); break;
    case 8: launch_any<8>(s, a, big, groups, (unsigned)grid); break;
    case 16: launch_any<16>(s, a, big, groups, (unsigned)grid); break;
    default: return DT_INVALID;
  }
  return launch_status();
}

}  // namespace dt
