// K3: ScaledDotProductAttention, flash-style, fp16 in / fp32 statistics, gfx950.
//
// One 512-thread workgroup (8 waves, two per SIMD) owns 256 query rows of one
// (batch, head); each wave owns 32 of them.  K/V arrive in tiles of 64 keys,
// transferred from memory straight into LDS, row-major (double-buffered, one
// barrier per tile).  Small launches take 128 rows, with two groups of waves
// that share out the key tiles (KG).
//
// Everything is computed transposed so that the query index is the MFMA
// column in every stage:
//   S^T = K Q^T          A = K tile rows from LDS, B = Q^T held in registers
//   O^T = V^T P^T        A = V^T, B = P^T = the S^T accumulators themselves
// With 32x32x16 MFMAs the column is lane & 31, and an accumulator holds rows
// 8*(v/4) + 4*(lane/32) + (v%4), v = 0..15.  With 16x16x32 MFMAs (M16) it is
// lane & 15 of two blocks of 16 queries, and an accumulator holds rows
// 4*(lane/16) + v, v = 0..3; those of 32 keys go side by side into one operand.
// Feeding accumulators back as the B operand only permutes the summation index,
// so the V^T operand is fetched with the same permutation and P never leaves
// registers; the softmax row reductions are in-lane plus exchanges between the
// lane groups of a column.  V stays row-major in LDS: the V^T operand (head
// dimension along lanes, keys along registers) comes from ds_read_b64_tr_b16,
// which hands lane j of a 16-lane group the element column (j % 4) of the rows
// addressed by lanes (j / 4) + {0, 4, 8, 12}.
//
// Which MFMA: for the same work 16x16x32 moves a fifth less through the register
// file, which counts where the launch is limited by the card's power, but leaves
// the exponentials of the SIMD's other wave 12 of every 16 issue clocks where
// 32x32x16 leaves 28 of 32 (an exponential takes 8: one to a slot, not three).
#include <algorithm>
#include <atomic>
#include <cstdlib>
#include <type_traits>

#include "dt_common.h"
#include "dt_qkprep.h"
#include "dt_sdpa.h"

namespace dt {

constexpr int BKV = 64;     // keys per tile
constexpr int WAVES = 8;    // waves per workgroup
// Query rows of a workgroup whose waves, 32 rows each, fall into `key_groups` groups (see sdpa_kernel).
constexpr int query_rows(int key_groups) { return WAVES / key_groups * 32; }
// Two key groups at head sizes up to 64 leave registers and LDS for two workgroups on a compute unit: four waves on a SIMD, of 128
// registers, which the loaders of several segments do not fit.
constexpr bool sdpa_four_waves(int dp, bool oneseg, int key_groups) { return dp == 64 && oneseg && key_groups == 2; }

typedef short short4_t __attribute__((ext_vector_type(4)));

__device__ __forceinline__ float fast_exp2(float x) { return __builtin_amdgcn_exp2f(x); }

// LDS layouts (measured bank-conflict free on this part: 64 banks, 16 lanes of
// a 16-byte access or 32 lanes of an 8-byte access per clock).
// K tile: [64 keys][DP] halfs; 16-byte chunk c of key row r is stored at a
// swizzled chunk so that 16 consecutive rows of one chunk column spread over
// all banks.
template <int DP>
__device__ __forceinline__ int k_chunk_swz(int row, int c) {
  if constexpr (DP == 128) return c ^ (row & 15);
  return c ^ ((row >> 1) & 7);
}
// V tile: [64 keys][DP] halfs; 32 lanes of the transposing read touch 4
// consecutive key rows x 64 contiguous bytes (M16: 8 x 32), so units of that
// many bytes are swizzled over the row index.
template <int DP, bool M16>
__device__ __forceinline__ int v_unit_swz(int row, int u) {
  static_assert(!M16 || DP == 128, "head sizes up to 64 are 32x32x16");
  if constexpr (M16) return u ^ (row & 7);
  return u ^ (DP == 128 ? row & 3 : (row >> 1) & 1);
}

// The lane groups of a wave -- two of 32, M16: four of 16 -- hold the same matrix columns: combine them without touching LDS.
__device__ __forceinline__ void halves16(float v, float& even, float& odd) {  // groups {0, 0, 2, 2} and {1, 1, 3, 3}
  uint32_t a = __builtin_bit_cast(uint32_t, v), b = a;
  asm volatile("" : "+v"(b));  // (as in halves32)
  auto r = __builtin_amdgcn_permlane16_swap(a, b, false, false);
  uint32_t x0 = r[0], x1 = r[1];
  asm volatile("" : "+v"(x0), "+v"(x1));
  even = __builtin_bit_cast(float, x0);
  odd = __builtin_bit_cast(float, x1);
}
template <bool M16>
__device__ __forceinline__ float max_groups(float v) {
  if constexpr (!M16) return max32(v);
  float a, b;
  halves16(v, a, b);
  return max32(fmaxf(a, b));
}
template <bool M16>
__device__ __forceinline__ float sum_groups(float v) {
  if constexpr (!M16) return sum32(v);
  float a, b;
  halves16(v, a, b);
  return sum32(a + b);
}

// KG: the waves of a workgroup fall into that many groups, which share the task's query rows and take every KG-th key tile each;
// two meet through LDS at the end.
// (VALU instructions of one wave run in the shadow of another's MFMAs only to a small degree, also with four waves on a SIMD: full
// rounds gain nothing by this, small launches the finer tasks.)
//
// SPLIT: for launches whose task count -- a task being the query rows of a workgroup, of one (batch, head) -- leaves the last round
// of workgroups mostly empty.  The first whole_tasks tasks, full rounds of them, go to a workgroup each; each of the
// others is cut along its keys into `shares` equal parts.  A workgroup with a part holds its unnormalised fp32 output,
// reference maximum and row sums, and the parts meet in pairs, the pairs in pairs, and so on: of two that meet, the
// first leaves what it holds in its workspace slot, counts itself in and ends; the other one folds it into its own
// registers and goes on to the next meeting, the last of them to the output.  Nobody waits for anybody, and the fold is
// the same whichever came first.  (Runs of several tasks' parts per workgroup, folded one after the other by the last
// to arrive, balance better on paper; that kernel needed 370 registers, and its spills made a tile 1.8 times as long.)
//
// M16: 16x16x32 MFMAs.  DL: head dimension that is multiplied (M16: D rounded up to a block of 16; DP, what a tile row
// holds, otherwise).
template <int DP, int DL, bool M16, bool PREMUL, bool ONESEG, bool SPLIT, int KG>
__global__ void __launch_bounds__(512, (sdpa_four_waves(DP, ONESEG, KG) ? 4 : 2)) sdpa_kernel(const SdpaArgs a) {
  constexpr bool FOUR = sdpa_four_waves(DP, ONESEG, KG);
  constexpr int QW = WAVES / KG;               // waves of a key group
  constexpr int QROWS = query_rows(KG);
  constexpr int ROWB = DP * 2;                 // bytes per tile row
  constexpr int TILE_B = BKV * ROWB;           // bytes of one K (or V) tile
  constexpr int LOADS = TILE_B / (QW * 1024);  // 16-byte chunks per thread per tile
  constexpr int LROWS = QW * 1024 / ROWB;      // rows of a tile that a load of all threads covers
  constexpr int MB = M16 ? 16 : 32;            // rows and columns of an MFMA
  constexpr int MK = M16 ? 32 : 16;            // its k-step
  constexpr int QB = 32 / MB;                  // its blocks in a wave's 32 queries
  constexpr int NV = M16 ? 4 : 16;             // its sums per lane
  constexpr int DB = (DL + MB - 1) / MB;       // its blocks of the head dimension
  constexpr int KS = (DL + MK - 1) / MK;       // k-steps over the head dimension
  typedef typename std::conditional<M16, float4_t, float16_t>::type sums_t;
  static_assert(!SPLIT || KG == 1, "tasks are cut with one key group");
  static_assert(LOADS >= 1 && LROWS % 16 == 0, "tile");

  // Two stages each for K and V: a tile is read from one while the next is in
  // flight into the other.
  __shared__ __attribute__((aligned(1024))) unsigned char Ks0[KG * TILE_B];
  __shared__ __attribute__((aligned(1024))) unsigned char Ks1[KG * TILE_B];
  __shared__ __attribute__((aligned(1024))) unsigned char Vs0[KG * TILE_B];
  __shared__ __attribute__((aligned(1024))) unsigned char Vs1[KG * TILE_B];

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = tid >> 6;
  const int qwave = wave & (QW - 1);                                      // which of the task's rows
  const int kg = KG == 1 ? 0 : __builtin_amdgcn_readfirstlane(wave / QW);  // key group
  const int col = lane & (MB - 1);  // row or column of an MFMA block
  const int grp = lane / MB;        // lane group: which k

  // XCD-aware order: tiles of one (batch, head) are consecutive, and each XCD
  // gets a contiguous run, so a head's K/V stay in one XCD's L2.
  auto xcd_order = [](int i, int total) __attribute__((always_inline)) {
    const int per = total / 8;
    return i < per * 8 ? (i & 7) * per + (i >> 3) : i;
  };
  // SPLIT: the first whole_tasks workgroups take a task each, bid counts the others
  int bid = blockIdx.x;
  const bool takes_whole = SPLIT && bid < a.whole_tasks;
  if constexpr (SPLIT) bid = takes_whole ? xcd_order(bid, a.whole_tasks) : xcd_order(bid - a.whole_tasks, a.total_blocks);
  else bid = xcd_order(bid, a.total_blocks);
  const int64_t Sq = a.Sq, Skv = a.Skv;
  const int D = a.D;
  const int n_tiles = (int)((Skv + BKV - 1) / BKV), full_tiles = (int)(Skv / BKV);

  // ---- per-thread constants of the K / V tile loaders ---------------------
  // Tiles go from memory straight into LDS.  A wave's transfer instruction
  // fills 1 KB of a tile, lane l landing on its 16-byte slot l; each thread
  // issues LOADS of them per K tile and per V tile and fetches the chunk that
  // the swizzle assigns to its slot.  Lanes whose chunk lies past D stay idle
  // (those slots keep the zeros they were given at the start), and so do, for
  // K, lanes whose row lies past the last key (their scores are masked whatever
  // the slot holds); V rows past the last key are zeroed (see zero_slot).
  // One key group: a wave's loads cover consecutive rows, each with an offset
  // in a register of its own.  Two, whose threads have twice as many: LROWS rows
  // apart, whose chunk is the same (the swizzles depend on row % 16 at most), at
  // one offset from bases that are.  (One offset costs one group 1 % of a launch.)
  constexpr int OFFS = KG == 1 ? LOADS : 1;
  const int qwave_u = __builtin_amdgcn_readfirstlane(qwave);
  int ld_row[LOADS], k_ch[LOADS], v_ch[LOADS];
  auto place = [](int w, int i) __attribute__((always_inline)) { return (KG == 1 ? w * LOADS + i : i * QW + w) * 1024; };
#pragma unroll
  for (int i = 0; i < LOADS; i++) {
    const int off = place(qwave, KG == 1 ? i : 0) + lane * 16;
    const int row = off / ROWB, pc = (off % ROWB) / 16;
    ld_row[i] = row + (KG == 1 ? 0 : i * LROWS);
    k_ch[i] = k_chunk_swz<DP>(row, pc);  // (the swizzles are involutions)
    v_ch[i] = M16 ? v_unit_swz<DP, M16>(row, pc >> 1) * 2 + (pc & 1) : v_unit_swz<DP, M16>(row, pc >> 2) * 4 + (pc & 3);
  }
  auto slot = [&](int i) __attribute__((always_inline)) { return (uint32_t)(kg * TILE_B + place(qwave_u, i)); };  // in a stage
  // slots that no transfer will ever write must not hold NaN patterns
  if (D < DP || Skv % BKV != 0) {
    for (int i = tid * 16; i < KG * TILE_B; i += 512 * 16) {
      *reinterpret_cast<uint4_t*>(Ks0 + i) = uint4_t{0, 0, 0, 0};
      *reinterpret_cast<uint4_t*>(Ks1 + i) = uint4_t{0, 0, 0, 0};
      *reinterpret_cast<uint4_t*>(Vs0 + i) = uint4_t{0, 0, 0, 0};
      *reinterpret_cast<uint4_t*>(Vs1 + i) = uint4_t{0, 0, 0, 0};
    }
    __syncthreads();
  }

  // ---- per-lane LDS read offsets --------------------------------------------
  // K operand: key row kb*MB + col, chunk of the group's 8 head-dim elements in k-step ks
  int k_rd[KS];
#pragma unroll
  for (int ks = 0; ks < KS; ks++) k_rd[ks] = kg * TILE_B + col * ROWB + k_chunk_swz<DP>(col, ks * (MK / 8) + grp) * 16;
  // V^T operand through the transposing read: lane i of a 16-lane group addresses key row (i / 4) of a 4-key run and 4
  // head-dim elements at 4 * (i % 4).  M16: the run is the group's, the elements those of block db.  Else: the run is the
  // half-wave's, and its two groups cover head-dim 0..15 and 16..31 of block db.
  const int li = lane & 15, dg = (lane >> 4) & 1;
  int v_rd[DB];
#pragma unroll
  for (int db = 0; db < DB; db++) {
    const int row = 4 * grp + (li >> 2);  // + multiples of 8 (M16: 16) per read: the swizzle depends on row & 3 (7) at most
    v_rd[db] = kg * TILE_B + row * ROWB + (M16 ? v_unit_swz<DP, M16>(row, db) * 32 : v_unit_swz<DP, M16>(row, db) * 64 + dg * 32) + (li & 3) * 8;
  }
  const float c = PREMUL ? 1.0f : a.scale_log2e;

  // ---- the work of this workgroup: key tiles [t_lo, t_hi) of a task, dealt out to its key groups -----
  int task = bid, t_lo = 0, t_hi = n_tiles, share = 0;
  if constexpr (SPLIT) {
    if (!takes_whole) {
      // part by part: the workgroups that run together on a die read the same keys of neighbouring tasks
      share = bid / a.cut_tasks;
      task = a.whole_tasks + (bid - share * a.cut_tasks);
      t_lo = (int)((int64_t)share * n_tiles / a.shares);
      t_hi = (int)((int64_t)(share + 1) * n_tiles / a.shares);
    }
  }
  const int t0 = t_lo + kg;                         // this group's first
  const int n_steps = (t_hi - t_lo + KG - 1) / KG;  // of the groups: the last one may be without a tile in its last step
  const int qt = task % a.q_tiles;
  const int bh = task / a.q_tiles;
  const int h = bh % a.Hq;
  const int b = bh / a.Hq;
  const int hk = h / a.group;

  // ---- Q^T fragments straight from global memory -----------------------
  // B operand of K Q^T: lane holds query column col of block qb, head-dim slots MK*ks + 8*grp + 0..7.  What the norm and the
  // rotation need is asked for together with the rows (one after the other, behind tests of each chunk's alignment, 24 x 2637 tokens
  // took 11 us for it), all of it ahead of what the loaders need, which hides the way to the rows: us, 24 heads of 64 / 128, 1344 tokens in
  // two segments, asked for behind it 28.9 / 39.7, here 28.6 / 39.3.  A lane's segment is an index into the arguments: selecting
  // among all eight takes some 0.6 us of arithmetic.
  half8_t qf[QB][KS];
  uint4_t raw[QB][KS], gam[QB][KS], rot[QB][KS];
  bool has_gam[QB];
  const auto chunk = [](const uint16_t* p, bool aligned) __attribute__((always_inline)) {
    if (aligned) return *reinterpret_cast<const uint4_t*>(p);  // uniform
    uint4_t v;
#pragma unroll
    for (int q = 0; q < 4; q++) v[q] = (uint32_t)p[2 * q] | ((uint32_t)p[2 * q + 1] << 16);
    return v;
  };
#pragma unroll
  for (int qb = 0; qb < QB; qb++) {
    int64_t qi = (int64_t)qt * QROWS + qwave * 32 + qb * MB + col;
    if (qi >= Sq) qi = Sq - 1;
    int sg = 0;
#pragma unroll
    for (int i = 1; i < kMaxSeg; i++)
      if (i < a.n_qseg && qi >= a.q[i].start) sg = i;
    const uint16_t* const qp = a.q[sg].ptr + b * a.q[sg].sb + (qi - a.q[sg].start) * a.q[sg].ss + h * a.q[sg].sh;
    const uint16_t* gp = a.q_gamma[sg];
    has_gam[qb] = gp != nullptr;
    if (!gp) gp = qp;  // (anything that can be read)
#pragma unroll
    for (int ks = 0; ks < KS; ks++) {
      const int d0 = ks * MK + grp * 8;
      raw[qb][ks] = gam[qb][ks] = rot[qb][ks] = uint4_t{0, 0, 0, 0};
      if (d0 < D) {
        raw[qb][ks] = *reinterpret_cast<const uint4_t*>(qp + d0);
        if (a.q_norm) gam[qb][ks] = chunk(gp + d0, a.q_aligned);  // uniform
        if (a.q_rot) rot[qb][ks] = chunk(a.q_rot + qi * D + d0, a.q_aligned);
      }
    }
  }

  // ---- K / V tile loaders ------------------------------------------------
  // ONESEG: K and V are one run of rows each and small enough for 32-bit byte
  // offsets from a uniform base; a tile step moves these (two key groups: that).
  // Otherwise the segment of a tile is looked up once per tile (uniformly): a
  // tile that lies inside one segment is fetched from that segment's base with
  // per-lane 32-bit offsets, a tile that straddles segments row by row.
  uint32_t k_off[OFFS], v_off[OFFS];  // of a thread's rows in a tile (of the first)
  const char* k_base = nullptr;
  const char* v_base = nullptr;
  uint32_t k_step = 0, v_step = 0;
  const int64_t keys_ahead = Skv - (int64_t)t0 * BKV;                        // keys from this group's first tile on
  int rows_left = (int)(keys_ahead < 0x7fffffff ? keys_ahead : 0x7fffffff);  // ONESEG: keys from the next K tile on
  int rows_left_v = rows_left;
  if constexpr (ONESEG) {
    k_step = (uint32_t)(a.k[0].ss * BKV * 2);
    v_step = (uint32_t)(a.v[0].ss * BKV * 2);
    k_base = reinterpret_cast<const char*>(a.k[0].ptr + b * a.k[0].sb + hk * a.k[0].sh) + (int64_t)t0 * k_step;
    v_base = reinterpret_cast<const char*>(a.v[0].ptr + b * a.v[0].sb + hk * a.v[0].sh) + (int64_t)t0 * v_step;
#pragma unroll
    for (int i = 0; i < OFFS; i++) {
      k_off[i] = (uint32_t)((ld_row[i] * a.k[0].ss + k_ch[i] * 8) * 2);
      v_off[i] = (uint32_t)((ld_row[i] * a.v[0].ss + v_ch[i] * 8) * 2);
    }
  }
  // General case: a uniform cursor holds the address of the group's next tile's first row, the step to its tile behind it and
  // the first tile that does not lie wholly inside the segment.  Up to there a tile costs one scalar comparison and one
  // addition, and its lanes fetch with 32-bit offsets from the cursor; from there on the cursor moves to the segment that the tile
  // starts in, and where that does not hold all of it -- the tile straddles segments or ends the sequence -- it goes row by row.
  struct SegCursor {
    const char* base;
    int64_t step;
    int rows;       // from a thread's row of a tile to its next
    int inside;  // tiles below this one lie inside the segment
  };
  auto seek = [&](const SdpaSeg* segs, SegCursor& c, uint32_t (&off)[OFFS], const int (&chs)[LOADS], int t)
                  __attribute__((always_inline)) {
    const int64_t row0 = (int64_t)t * BKV;
    int sg = 0;
#pragma unroll
    for (int i = 1; i < kMaxSeg; i++)
      if (i < a.n_kvseg && row0 >= segs[i].start) sg = i;
    sg = __builtin_amdgcn_readfirstlane(sg);  // (comparisons of 64 bits leave uniform values in vector registers)
    const int64_t ss = segs[sg].ss, end = (sg + 1 < a.n_kvseg) ? segs[sg + 1].start : Skv;
    c.inside = __builtin_amdgcn_readfirstlane(ss > 0 && ss < (1 << 24) ? (int)(end / BKV) : 0);
    c.step = ss * (KG * BKV * 2);
    c.rows = (int)(ss * (LROWS * 2));  // (where `inside` says that the cursor is used)
    c.base = reinterpret_cast<const char*>(segs[sg].ptr + b * segs[sg].sb + hk * segs[sg].sh + (row0 - segs[sg].start) * ss);
#pragma unroll
    for (int i = 0; i < OFFS; i++) off[i] = (uint32_t)((ld_row[i] * ss + chs[i] * 8) * 2);
  };
  SegCursor kcur{}, vcur{};
  if constexpr (!ONESEG) {
    seek(a.k, kcur, k_off, k_ch, t0);
    seek(a.v, vcur, v_off, v_ch, t0);
  }
  // (zero_tail: rows of the tile past the last key get zeros instead of keeping an earlier tile's bytes -- for V,
  // whose stale rows would otherwise meet a probability of exactly zero in the second MFMA: 0 x Inf = NaN)
  // What the paths that few tiles take derive from a thread's place is not to be kept in registers across the loop: they are short
  // with four waves on a SIMD, and a reload from scratch waits for the transfers in flight.  (Nine registers at head sizes over 48 and four
  // below do go to scratch; they come back behind the loop and where a ragged tile's rows are zeroed, nowhere else.)
  auto opaque = [](int v) __attribute__((always_inline)) {
    if constexpr (FOUR) asm volatile("" : "+v"(v));
    return v;
  };
  auto zero_slot = [&](unsigned char* dst, int i) __attribute__((always_inline)) {
    *reinterpret_cast<uint4_t*>(dst + slot(i) + opaque(lane) * 16) = uint4_t{0, 0, 0, 0};
  };
  auto issue_general = [&](const SdpaSeg* segs, SegCursor& c, uint32_t (&off)[OFFS], const int (&chs)[LOADS],
                           unsigned char* dst, int t, bool zero_tail) __attribute__((always_inline)) {
    if (t >= c.inside && t < full_tiles) seek(segs, c, off, chs, t);  // uniform
    if (t < c.inside) {                                               // uniform
      const int64_t rows = KG == 1 ? 0 : __builtin_amdgcn_readfirstlane(c.rows);
#pragma unroll
      for (int i = 0; i < LOADS; i++)
        if (chs[i] * 8 < D) load_to_lds_16(c.base + i * rows, off[KG == 1 ? i : 0], lds_address(dst) + slot(i));
      c.base += c.step;
      return;
    }
    const int64_t row0 = (int64_t)t * BKV;
#pragma unroll
    for (int i = 0; i < LOADS; i++) {
      const int64_t kj = row0 + ld_row[i];
      if (kj >= Skv) {
        if (zero_tail) zero_slot(dst, i);
      } else if (chs[i] * 8 < D) {
        int sl = 0;
#pragma unroll
        for (int u = 1; u < kMaxSeg; u++)
          if (u < a.n_kvseg && kj >= segs[u].start) sl = u;
        const uint16_t* src =
            segs[sl].ptr + b * segs[sl].sb + (kj - segs[sl].start) * segs[sl].ss + hk * segs[sl].sh + chs[i] * 8;
        load_to_lds_16(src, lds_address(dst) + slot(i));
      }
    }
  };
  auto advance = [](const char*& base, uint32_t (&off)[OFFS], uint32_t step) __attribute__((always_inline)) {
    if constexpr (KG > 1) base += (int64_t)KG * step;
    else {
#pragma unroll
      for (int i = 0; i < OFFS; i++) off[i] += step;
    }
  };
  // starts the transfer of the group's next K (or V) tile and moves on to the one behind it
  auto issue_k = [&](unsigned char* dst, [[maybe_unused]] int t) __attribute__((always_inline)) {
    if constexpr (ONESEG) {
#pragma unroll
      for (int i = 0; i < LOADS; i++)
        if (ld_row[i] < rows_left && k_ch[i] * 8 < D)
          load_to_lds_16(k_base + (KG == 1 ? 0 : (int64_t)i * (k_step / BKV * LROWS)), k_off[KG == 1 ? i : 0], lds_address(dst) + slot(i));
      advance(k_base, k_off, k_step);
      rows_left -= KG * BKV;
    } else {
      issue_general(a.k, kcur, k_off, k_ch, dst, t, false);
    }
  };
  auto issue_v = [&](unsigned char* dst, [[maybe_unused]] int t) __attribute__((always_inline)) {
    if constexpr (ONESEG) {
      if (rows_left_v < BKV) {  // uniform: the ragged last tile
#pragma unroll
        for (int i = 0; i < LOADS; i++)
          if (ld_row[i] >= rows_left_v) zero_slot(dst, i);
      }
#pragma unroll
      for (int i = 0; i < LOADS; i++)
        if (ld_row[i] < rows_left_v && v_ch[i] * 8 < D)
          load_to_lds_16(v_base + (KG == 1 ? 0 : (int64_t)i * (v_step / BKV * LROWS)), v_off[KG == 1 ? i : 0], lds_address(dst) + slot(i));
      advance(v_base, v_off, v_step);
      rows_left_v -= KG * BKV;
    } else {
      issue_general(a.v, vcur, v_off, v_ch, dst, t, true);
    }
  };
  // ---- the queries' norm and rotation --------------------------------------
#pragma unroll
  for (int qb = 0; qb < QB; qb++) {
    if (a.q_prep) {  // uniform
      // RMSNorm over the head, then the rotation: the row's D elements sit in the lanes of this column
      float inv = 1.f;
      if (a.q_norm) {  // uniform: some segment has a norm weight, and the sum takes every lane
        float ss = 0.f;
#pragma unroll
        for (int ks = 0; ks < KS; ks++) {
          float x[8];
          unpack_chunk(raw[qb][ks], x);
#pragma unroll
          for (int e = 0; e < 8; e++) ss += x[e] * x[e];
        }
        ss = sum_groups<M16>(ss);
        if (has_gam[qb]) inv = 1.0f / sqrtf(ss / (float)D + a.q_eps);
      }
#pragma unroll
      for (int ks = 0; ks < KS; ks++) {
        float x[8];
        unpack_chunk(raw[qb][ks], x);
        raw[qb][ks] = finish_chunk(x, inv, has_gam[qb], gam[qb][ks], a.q_rot != nullptr, rot[qb][ks], 1.0f);
      }
    }
#pragma unroll
    for (int ks = 0; ks < KS; ks++) qf[qb][ks] = __builtin_bit_cast(half8_t, raw[qb][ks]);
  }

  // ---- running state -----------------------------------------------------
  sums_t oacc[DB][QB];  // O^T: [block of the head dimension][block of queries]
#pragma unroll
  for (int db = 0; db < DB; db++)
#pragma unroll
    for (int qb = 0; qb < QB; qb++)
#pragma unroll
      for (int v = 0; v < NV; v++) oacc[db][qb][v] = 0.f;
  float m_ref[QB];  // reference for the exponentials (raw score units); trails the true running maximum
  float l_run[QB];  // this lane's share of the row sums
#pragma unroll
  for (int qb = 0; qb < QB; qb++) {
    m_ref[qb] = -INFINITY;
    l_run[qb] = 0.f;
  }

  constexpr int KB = BKV / MB;        // blocks of keys in a tile
  constexpr int PK = M16 ? 32 : 16;   // keys of a second MFMA
  sums_t sacc[KB][QB];                // S^T of the tile in flight: [block of keys][block of queries]
  half8_t pf[BKV / PK][QB];           // its probabilities, as the B operand of the second MFMA
  auto mfma = [](half8_t a, half8_t b, sums_t sum) __attribute__((always_inline)) {
    if constexpr (M16) return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, sum, 0, 0, 0);
    else return __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, sum, 0, 0, 0);
  };

  // S^T = K Q^T for the K tile in stage st
  auto s_phase = [&](const unsigned char* kt) __attribute__((always_inline)) {
#pragma unroll
    for (int kb = 0; kb < KB; kb++)
#pragma unroll
      for (int qb = 0; qb < QB; qb++)
#pragma unroll
        for (int v = 0; v < NV; v++) sacc[kb][qb][v] = 0.f;
    if constexpr (FOUR) {  // (the waves hide the reads for each other)
#pragma unroll
      for (int ks = 0; ks < KS; ks++) {
#pragma unroll
        for (int kb = 0; kb < KB; kb++)
          sacc[kb][0] = mfma(*reinterpret_cast<const half8_t*>(kt + kb * MB * ROWB + k_rd[ks]), qf[0][ks], sacc[kb][0]);
        if (ks & 1) __builtin_amdgcn_sched_barrier(0);
      }
      __builtin_amdgcn_sched_barrier(0);
      return;
    }
    // K fragments are read a group of four ahead of the MFMAs that use them: KB blocks of 4 / KB k-steps
    constexpr int GS = 4 / KB;
    half8_t kf[2][4];
    // (A k-step that lies wholly in the zero padding of a head size is left out.  One key group tests for it at all head sizes up to
    // 64: where no k-step does, the loop is 7 % slower without the branches, and at 40 a kernel that knows is no faster -- us, 2 x 10 x 4096 of 64
    // 143 / 154, 2 x 8 x 4096 of 40 74.4 / 74.6, 24 x 1344 of 40 26.6 / 27.3.)
    auto live = [&](int ks) __attribute__((always_inline)) { return M16 || DL != 64 || ks * MK < D; };
    auto read_k = [&](int buf, int g) __attribute__((always_inline)) {
#pragma unroll
      for (int u = 0; u < 4; u++) {
        const int ks = g * GS + u / KB, kb = u % KB;
        if (ks < KS && live(ks)) kf[buf][u] = *reinterpret_cast<const half8_t*>(kt + kb * MB * ROWB + k_rd[ks < KS ? ks : 0]);
      }
    };
    read_k(0, 0);
#pragma unroll
    for (int g = 0; g * GS < KS; g++) {
      __builtin_amdgcn_sched_barrier(0);
      if ((g + 1) * GS < KS) read_k((g + 1) & 1, g + 1);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int u = 0; u < 4; u++) {
        const int ks = g * GS + u / KB, kb = u % KB;
        if (ks < KS && live(ks)) {
#pragma unroll
          for (int qb = 0; qb < QB; qb++) sacc[kb][qb] = mfma(kf[g & 1][u], qf[qb][ks < KS ? ks : 0], sacc[kb][qb]);
        }
      }
    }
    __builtin_amdgcn_sched_barrier(0);
  };

  // online softmax of tile t (per query column, statistics in fp32): sacc -> pf
  auto softmax_phase = [&](int t) __attribute__((always_inline)) {
    const int rem = (int)(Skv - (int64_t)t * BKV);  // keys left, this tile included
    const bool ragged = rem < BKV;
    if (PREMUL || ragged) {
#pragma unroll
      for (int kb = 0; kb < KB; kb++)
#pragma unroll
        for (int qb = 0; qb < QB; qb++)
#pragma unroll
          for (int v = 0; v < NV; v++) {
            float s = sacc[kb][qb][v];
            if (PREMUL) s *= a.scale_log2e;
            if (ragged) {
              const int kj = kb * MB + 8 * (v >> 2) + 4 * grp + (v & 3);
              if (kj >= rem) s = -INFINITY;
            }
            sacc[kb][qb][v] = s;
          }
    }
    // Probabilities against the current reference, and this lane's share of their row sums.  The tile's maximum is
    // not looked for: as long as every lane's sums stay below 2^10 no probability exceeds that (fp16 holds 2^16),
    // which is all that the reference is there to ensure.  (The sums are of the fp32 probabilities at every head size.  A column of
    // ones in V's padding, which has the second MFMA add up the fp16 ones, is 3 us of 72 faster at 2 x 8 heads of 40, 4096 x 4096, and
    // loses what lies below 2^-25 of the reference: 16383 such keys beside one took a result from 0.9995 to 1.)
    float psum[QB];
    auto probabilities = [&]() __attribute__((always_inline)) {
      float mc[QB];
#pragma unroll
      for (int qb = 0; qb < QB; qb++) {
        mc[qb] = m_ref[qb] * c;
        psum[qb] = 0.f;
      }
#pragma unroll
      for (int kb = 0; kb < KB; kb++)
#pragma unroll
        for (int v = 0; v < NV; v++)
#pragma unroll
          for (int qb = 0; qb < QB; qb++) {
            const float p = fast_exp2(__builtin_fmaf(sacc[kb][qb][v], c, -mc[qb]));
            psum[qb] += p;
            const int slot = kb * NV + v;  // of this lane's scores: eight to an operand
            pf[slot >> 3][qb][slot & 7] = (half_t)p;
            if constexpr (FOUR)  // (operand by operand: 128 registers hold no more than one operand's probabilities in fp32)
              if ((slot & 7) == 7) __builtin_amdgcn_sched_barrier(0);
          }
    };
    probabilities();
    // (the first tile arrives here with the references at -inf: its sums are inf; a NaN fails the test too)
    bool outgrown = !(psum[0] <= 1024.0f);
    if constexpr (QB == 2) outgrown = outgrown || !(psum[1] <= 1024.0f);
    if (__builtin_amdgcn_ballot_w64(outgrown) != 0) {
      // some row's scores have outgrown the reference: move every row's reference up to its running maximum,
      // rescale what has been accumulated, and redo this tile's probabilities
#pragma unroll
      for (int qb = 0; qb < QB; qb++) {
        float mx = sacc[0][qb][0];
#pragma unroll
        for (int kb = 0; kb < KB; kb++)
#pragma unroll
          for (int v = (kb == 0 ? 1 : 0); v < NV; v++) mx = fmaxf(mx, sacc[kb][qb][v]);
        mx = max_groups<M16>(mx);
        // (Finite even where every score so far is -inf -- keys masked through the dot product itself: against a
        // reference of -inf the probabilities would be NaN, in a part of the keys that counts for nothing.  No finite
        // score lies below: |q k| <= 128 * 65504^2 = 5.5e11, and PREMUL's own scale has the whole range of fp32.)
        const float m_new = fmaxf(fmaxf(m_ref[qb], mx), PREMUL ? -3e38f : -1e12f);
        const float alpha = fast_exp2((m_ref[qb] - m_new) * c);  // first tile: exp2(-inf) = 0
        m_ref[qb] = m_new;
        l_run[qb] *= alpha;
#pragma unroll
        for (int db = 0; db < DB; db++)
#pragma unroll
          for (int v = 0; v < NV; v++) oacc[db][qb][v] *= alpha;
      }
      probabilities();
    }
#pragma unroll
    for (int qb = 0; qb < QB; qb++)
      l_run[qb] += psum[qb];
  };

  // O^T += V^T P^T for the V tile in stage st.
  // k-slot e of lane group grp in step s of PK keys is key PK*s + (PK/2)*(e/4) + 4*grp + (e%4).
  auto pv_phase = [&](const unsigned char* vt) __attribute__((always_inline)) {
    typedef __attribute__((address_space(3))) short4_t lds_s4;
    typedef short short8_t __attribute__((ext_vector_type(8)));
    if constexpr (FOUR) {
#pragma unroll
      for (int s = 0; s < BKV / PK; s++) {
        if (s % 2 == 0) __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int db = 0; db < DB; db++) {
          const short4_t lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s4*)(vt + PK * s * ROWB + v_rd[db]));
          const short4_t h4 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s4*)(vt + (PK * s + PK / 2) * ROWB + v_rd[db]));
          oacc[db][0] = mfma(__builtin_bit_cast(half8_t, short8_t{lo[0], lo[1], lo[2], lo[3], h4[0], h4[1], h4[2], h4[3]}), pf[s][0], oacc[db][0]);
        }
      }
      __builtin_amdgcn_sched_barrier(0);
      return;
    }
    // V^T fragments (DB blocks per step) go in groups of up to four, the next group read while the current one's MFMAs run
    constexpr int GF = M16 ? 4 : DB, NF = BKV / PK * DB, NG = (NF + GF - 1) / GF;
    short4_t vlo[2][GF], vhi[2][GF];
    auto read_v = [&](int buf, int g) __attribute__((always_inline)) {
#pragma unroll
      for (int u = 0; u < GF; u++) {
        const int f = g * GF + u, koff = PK * (f / DB) * ROWB;
        if (f >= NF) continue;
        vlo[buf][u] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s4*)(vt + koff + v_rd[f % DB]));
        vhi[buf][u] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s4*)(vt + koff + PK / 2 * ROWB + v_rd[f % DB]));
      }
    };
    read_v(0, 0);
#pragma unroll
    for (int g = 0; g < NG; g++) {
      __builtin_amdgcn_sched_barrier(0);
      if (g + 1 < NG) read_v((g + 1) & 1, g + 1);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int u = 0; u < GF; u++) {
        const int f = g * GF + u;
        if (f >= NF) continue;
        const short4_t lo = vlo[g & 1][u], h4 = vhi[g & 1][u];
        const short8_t v8 = short8_t{lo[0], lo[1], lo[2], lo[3], h4[0], h4[1], h4[2], h4[3]};
#pragma unroll
        for (int qb = 0; qb < QB; qb++)
          oacc[f % DB][qb] = mfma(__builtin_bit_cast(half8_t, v8), pf[f / DB][qb], oacc[f % DB][qb]);
      }
    }
    __builtin_amdgcn_sched_barrier(0);
  };

  // ---- pipeline ---------------------------------------------------------------
  if (t0 < t_hi) {  // uniform
    issue_k(Ks0, t0);
    if constexpr (FOUR) issue_v(Vs0, t0);
  }
  __builtin_amdgcn_s_waitcnt(0x0f70);  // vmcnt(0): this wave's part of the tiles has landed
  __syncthreads();
  if constexpr (FOUR) {
    // Step n (between two barriers) has the group's n-th K and V tiles readable in LDS while the next ones are written.  Four
    // waves share a SIMD, and what one of them waits for -- the MFMA pipe, an exponential, LDS -- the others fill.
    auto step = [&](int n, unsigned char* k_cur, unsigned char* k_next, unsigned char* v_cur, unsigned char* v_next)
                    __attribute__((always_inline)) {
      const int t = t0 + n * KG;
      if (t + KG < t_hi) {
        issue_k(k_next, t + KG);
        issue_v(v_next, t + KG);
      }
      if (t < t_hi) {
        s_phase(k_cur);
        softmax_phase(t);
        pv_phase(v_cur);
      }
      __builtin_amdgcn_s_waitcnt(0x0f70);
      __syncthreads();
    };
    for (int n = 0; n < n_steps; n += 2) {
      step(n, Ks0, Ks1, Vs0, Vs1);
      if (n + 1 < n_steps) step(n + 1, Ks1, Ks0, Vs1, Vs0);
    }
  } else {
    // Interval n (between two barriers) has K tile n and V tile n-1 of the group readable in
    // LDS while K tile n+1 and V tile n are written.  Every wave runs
    //   O += V(n-1) P(n-1) ;  S(n) = K(n) Q ;  P(n) = softmax(S(n))
    // per interval -- two MFMA phases back to back, then one VALU phase.  The two
    // waves of a SIMD (w and w+4) run that cycle half a period apart: the second
    // one starts each interval with the softmax of the scores it produced in the
    // previous interval, so one wave's exponentials overlap the other's MFMAs.
    const bool second = wave >= 4;
    // K(n) is in k_cur, V(n-1) in v_prev; K(n+1) goes to k_next, V(n) to v_cur
    auto interval = [&](int n, const unsigned char* k_cur, unsigned char* k_next, const unsigned char* v_prev,
                        unsigned char* v_cur) __attribute__((always_inline)) {
      const int t = t0 + n * KG;
      if (t + KG < t_hi) issue_k(k_next, t + KG);
      if (t < t_hi) issue_v(v_cur, t);
      // (with scalar loads of the segments' places on their way, which may come out of order, the compiler would wait for all LDS
      // reads in place of the next one: 3 % of a launch)
      if constexpr (!ONESEG) __builtin_amdgcn_s_waitcnt(0xc07f);  // lgkmcnt(0)
      const bool before = n > 0 && (KG == 1 || t - KG < t_hi);  // there is a tile n - 1
      // the wave doing softmax arithmetic gets issue priority: its exponentials only make progress in
      // the gaps the other wave's MFMA stream leaves (measured: +1 %; the opposite assignment -2 %)
      if (!second) {
        __builtin_amdgcn_s_setprio(0);
        if (before) pv_phase(v_prev);
        if (t < t_hi) {
          s_phase(k_cur);
          __builtin_amdgcn_s_setprio(2);
          softmax_phase(t);
        }
      } else {
        if (before) {
          __builtin_amdgcn_s_setprio(2);
          softmax_phase(t - KG);
          __builtin_amdgcn_s_setprio(0);
          pv_phase(v_prev);
        }
        if (t < t_hi) s_phase(k_cur);
      }
      __builtin_amdgcn_s_waitcnt(0x0f70);
      __syncthreads();
    };
    for (int n = 0; n <= n_steps; n += 2) {
      interval(n, Ks0, Ks1, Vs1, Vs0);
      if (n + 1 <= n_steps) interval(n + 1, Ks1, Ks0, Vs0, Vs1);
    }
    __builtin_amdgcn_s_setprio(0);
  }

  // the row sums, the same in every group of lanes from here on
#pragma unroll
  for (int qb = 0; qb < QB; qb++) l_run[qb] = sum_groups<M16>(l_run[qb]);

  // Where two hold partial results of the same rows, meet() takes in the other's reference and row sums and says how its sums are
  // folded: mine a + got b with both products rounded, the same for either order.
  struct Weights {
    float a, b;
    __device__ __forceinline__ float fold(float mine, float got) const {
      float x = mine * a, y = got * b;
      asm volatile("" : "+v"(x), "+v"(y));
      return x + y;
    }
  };
  auto meet = [&](int qb, float m_o, float l_o) __attribute__((always_inline)) {
    const float m_new = fmaxf(m_ref[qb], m_o);
    const Weights w{fast_exp2((m_ref[qb] - m_new) * c), fast_exp2((m_o - m_new) * c)};
    m_ref[qb] = m_new;
    l_run[qb] = w.fold(l_run[qb], l_o);
    return w;
  };
  constexpr int SUMS = DB * QB * NV;  // of a lane
  if constexpr (KG == 2) {
    // the second key group hands its results to the first through the tiles' LDS (the loop ended with a barrier)
    constexpr int QS = SUMS / 4;  // a quarter of the sums into each array
    static_assert(SUMS % 4 == 0 && QS * 4 * 64 * QW <= KG * TILE_B, "room");
    __shared__ float stats[QW][2 * QB][64];
    float* const quarter[4] = {reinterpret_cast<float*>(Ks0), reinterpret_cast<float*>(Ks1), reinterpret_cast<float*>(Vs0), reinterpret_cast<float*>(Vs1)};
    const int at = qwave * (QS * 64) + lane;
    if (kg == 1) {
#pragma unroll
      for (int i = 0; i < SUMS; i++) quarter[i / QS][at + i % QS * 64] = oacc[i / (QB * NV)][i / NV % QB][i % NV];
#pragma unroll
      for (int qb = 0; qb < QB; qb++) {
        stats[qwave][2 * qb][lane] = m_ref[qb];
        stats[qwave][2 * qb + 1][lane] = l_run[qb];
      }
    }
    __syncthreads();
    if (kg == 0) {
      Weights w[QB];
#pragma unroll
      for (int qb = 0; qb < QB; qb++) w[qb] = meet(qb, stats[qwave][2 * qb][lane], stats[qwave][2 * qb + 1][lane]);
#pragma unroll
      for (int i = 0; i < SUMS; i++) {
        sums_t& o = oacc[i / (QB * NV)][i / NV % QB];
        o[i % NV] = w[i / NV % QB].fold(o[i % NV], quarter[i / QS][at + i % QS * 64]);
      }
    } else {
      return;
    }
  }

  // ---- normalise and store O ----------------------------------------------
  // Runs of 8 consecutive head-dim elements per lane (16-byte stores) out of its runs of four: 32x32 blocks hold head-dim
  // 8*g + 4*grp + (0..3), and swapping the odd groups g of the low half-wave with the even ones of the high half-wave does
  // it; 16x16 blocks hold 4*grp + (0..3), and the odd lane groups of one block are swapped with the even ones of the next.
  auto store_output = [&]() __attribute__((always_inline)) {
    const bool vec_ok = ((a.o_sb | a.o_ss | a.o_sh) & 7) == 0 && (reinterpret_cast<uintptr_t>(a.o) & 15) == 0;
#pragma unroll
    for (int qb = 0; qb < QB; qb++) {
      const int64_t qi = (int64_t)qt * QROWS + qwave * 32 + qb * MB + col;
      const float inv = 1.0f / l_run[qb];
      uint16_t* op = a.o + b * a.o_sb + (qi < Sq ? qi : 0) * a.o_ss + h * a.o_sh;
      constexpr int RUNS = DB * NV / 4;  // this lane's runs of four
#pragma unroll
      for (int r = 0; r < RUNS; r += 2) {
        uint32_t pk[2][2];
#pragma unroll
        for (int u = 0; u < 2; u++)
#pragma unroll
          for (int e = 0; e < 2; e++) {
            const int n = (r + u < RUNS ? r + u : r) * 4 + 2 * e;  // (past the last block: never stored)
            pk[u][e] = (uint32_t)half_to_bits((half_t)(oacc[n / NV][qb][n % NV] * inv)) |
                       ((uint32_t)half_to_bits((half_t)(oacc[n / NV][qb][n % NV + 1] * inv)) << 16);
          }
        uint32_t run[4];
#pragma unroll
        for (int e = 0; e < 2; e++) {
          uint32_t x = pk[0][e], y = pk[1][e];
          if constexpr (RUNS % 2) asm volatile("" : "+v"(y));  // (the swap needs two distinct registers)
          auto got = M16 ? __builtin_amdgcn_permlane16_swap(x, y, false, false) : __builtin_amdgcn_permlane32_swap(x, y, false, false);
          run[e] = got[0];
          run[2 + e] = got[1];
        }
        const int d0 = M16 ? (r + (grp & 1)) * 16 + 8 * (grp >> 1) : r * 8 + 8 * grp;
        if (qi < Sq && d0 < D && (M16 ? r + (grp & 1) < RUNS : true)) {
          if (vec_ok) {
            *reinterpret_cast<uint4_t*>(op + d0) = uint4_t{run[0], run[1], run[2], run[3]};
          } else {
            *reinterpret_cast<uint2_t*>(op + d0) = uint2_t{run[0], run[1]};
            *reinterpret_cast<uint2_t*>(op + d0 + 4) = uint2_t{run[2], run[3]};
          }
        }
      }
    }
  };

  if constexpr (SPLIT) {
    if (!takes_whole) {
      __shared__ int s_seen;
      // Slot layout (floats): [DP / 2 accumulators][512 threads] (those past DL unused), then [512]: for a wave, the
      // reference maxima of its 32 queries and their row sums.  A wave's access covers 256 consecutive bytes.  The parts of a task run on any compute units of the
      // device, whose L2 caches (one per die) do not see each other's ordinary stores: slots are written and read with
      // device-scope accesses (relaxed atomics: write-through stores, loads that do not trust a die's cached copy)
      // instead of bracketing ordinary accesses with cache-wide write-backs and invalidations, which cost far more than
      // the 130 KB they would protect.
      constexpr int SLOT_F = sdpa_split_slot_floats(DP);
      const int cut = task - a.whole_tasks;
      float* const slots = a.partials + (size_t)cut * SLOT_F + tid;
      const size_t slot_step = (size_t)a.cut_tasks * SLOT_F;
      int32_t* const counters = a.counters + cut * kSdpaSplitNodes;
      int node0 = 0;  // counters of this level
      for (int level = 0; (1 << level) < a.shares; level++) {
        const int me = share >> level, other = me ^ 1;
        if ((other << level) < a.shares) {  // uniform; otherwise nobody to meet on this level
          int32_t* const met = counters + node0 + (me >> 1);
          if (tid == 0) s_seen = __hip_atomic_load(met, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
          __syncthreads();
          if (s_seen == 0) {  // uniform: the other one is not there yet
            float* const own = slots + (me << level) * slot_step;
#pragma unroll
            for (int db = 0; db < DB; db++)
#pragma unroll
              for (int qb = 0; qb < QB; qb++)
#pragma unroll
                for (int v = 0; v < NV; v++)
                  __hip_atomic_store(own + ((db * QB + qb) * NV + v) * 512, oacc[db][qb][v], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            const float stat = lane & 32 ? (grp & (QB - 1) ? l_run[QB - 1] : l_run[0]) : (grp & (QB - 1) ? m_ref[QB - 1] : m_ref[0]);
            __hip_atomic_store(own + DP / 2 * 512, stat, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            // every wave's stores have been acknowledged before the barrier, hence before the count that publishes them
            __builtin_amdgcn_s_waitcnt(0x0f70);  // vmcnt(0)
            __syncthreads();
            if (tid == 0) s_seen = __hip_atomic_fetch_add(met, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            __syncthreads();
            if (s_seen == 0) return;  // uniform: the other one goes on
          }
          const float* const theirs = slots + (other << level) * slot_step;
          auto ld = [&](int i) __attribute__((always_inline)) {
            return __hip_atomic_load(theirs + i, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
          };
          // (theirs is this thread's place: - lane + col is its column's in the first group of lanes)
          const int stats = DP / 2 * 512 - lane + col;
#pragma unroll
          for (int qb = 0; qb < QB; qb++) {
            const Weights w = meet(qb, ld(stats + MB * qb), ld(stats + 32 + MB * qb));
            constexpr int AT = 16 / NV;  // blocks whose sums are asked for together
#pragma unroll
            for (int d0 = 0; d0 < DB; d0 += AT) {
              sums_t got[AT];
#pragma unroll
              for (int u = 0; u < AT; u++)
                if (d0 + u < DB)
#pragma unroll
                  for (int v = 0; v < NV; v++) got[u][v] = ld((((d0 + u) * QB + qb) * NV + v) * 512);
#pragma unroll
              for (int u = 0; u < AT; u++)
                if (d0 + u < DB)
#pragma unroll
                  for (int v = 0; v < NV; v++) oacc[d0 + u][qb][v] = w.fold(oacc[d0 + u][qb][v], got[u][v]);
            }
          }
          __syncthreads();  // s_seen may be written again
        }
        node0 += kSdpaSplitNodes >> (level + 1);
      }
    }
  }
  store_output();
}

// Zeroes the counters of a SPLIT launch (a fill kernel, so that the launch can be captured in a graph).
__global__ void sdpa_zero_counters_kernel(int32_t* counters, int n) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) counters[i] = 0;
}

// Compute units of the calling thread's current device (cached per ordinal; 256 if the runtime cannot say).
static int compute_units() {
  static std::atomic<int> cached[64];
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess) {
    (void)hipGetLastError();
    return 256;
  }
  if (dev < 0 || dev >= 64) return 256;
  int n = cached[dev].load(std::memory_order_relaxed);
  if (n == 0) {
    if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || n <= 0) {
      (void)hipGetLastError();
      n = 256;
    }
    cached[dev].store(n, std::memory_order_relaxed);
  }
  return n;
}

bool sdpa_split_plan(int32_t B, int32_t Hq, int32_t D, int64_t Sq, int64_t Skv, SdpaSplit* plan) {
  if (B <= 0 || Hq <= 0 || D <= 0 || Sq <= 0 || Skv <= 0) return false;
  // DT_SDPA_KEY_SPLIT = "never" | "always" (whenever the launch can be cut at all; for tests and measurements);
  // anything else, or unset: decide by the estimate below.  Read at every call.
  const char* knob = getenv("DT_SDPA_KEY_SPLIT");
  const bool never = knob && knob[0] == 'n', always = knob && knob[0] == 'a';
  if (never) return false;
  const int64_t tasks = (int64_t)B * Hq * ((Sq + query_rows(1) - 1) / query_rows(1));
  const int64_t n_tiles = (Skv + BKV - 1) / BKV;
  if (tasks > (1 << 20) || tasks * n_tiles >= (1LL << 31)) return false;  // (the kernel counts units in 32 bits)
  const int cus = compute_units();
  const int64_t whole = tasks / cus * cus, cut = tasks - whole;  // full rounds of tasks, and what is left
  // as many parts per task as the round takes (of at least two key tiles)
  int64_t shares = cut > 0 ? cus / cut : 0;
  if (shares > kSdpaSplitNodes) shares = kSdpaSplitNodes;
  if (shares > n_tiles / 2) shares = n_tiles / 2;
  if (always && shares < 2 && n_tiles >= 2) shares = 2;
  if (cut == 0 || shares < 2) return false;
  if (!always) {
    // (launches of six rounds and more keep asking for no workspace: a seventh of their time at most is the last round)
    if (tasks >= 6LL * cus) return false;
    // Measured on this part: a key tile of the last, partial round takes 1.4 us at head size 128 (1.0 at 64 and below)
    // while most of the card idles and 1.9 us (1.2) when none of it does, and cutting costs 20 us (12): the counters'
    // launch, the parts' way out and in.  Head size 128, us before / after: 264 tasks of 42 key tiles 150 / 120, of 72
    // 244 / 181; 320 of 72 244 / 208; 384 of 42 151 / 150 (not cut); 64 of 72 98 / 64.  Head size 64: 264 of 42 100 / 77,
    // 64 of 72 72 / 42; 384 of 18 49 / 51 (not cut).
    const bool small = D <= 64;
    const double idle = small ? 1.0 : 1.4, full = small ? 1.2 : 1.9, fixed = small ? 12.0 : 20.0;
    const double busy = (double)(cut * shares) / cus;
    const double cut_time = (double)((n_tiles + shares - 1) / shares) * (idle + (full - idle) * busy) + fixed;
    if ((double)n_tiles * idle < cut_time + 4.0) return false;
  }
  if (plan) {
    plan->shares = (int32_t)shares;
    plan->cut_tasks = (int32_t)cut;
    plan->whole_tasks = (int32_t)whole;
    plan->counter_bytes = ((size_t)cut * kSdpaSplitNodes * 4 + 255) & ~(size_t)255;
    const size_t slot = (size_t)sdpa_split_slot_floats(D <= 64 ? 64 : 128) * 4;
    plan->partial_bytes = (size_t)(cut * shares) * slot;
    // What callers are asked to bring.  With full rounds in front: what the parts take (24 heads x 2637 tokens: 9 MB).
    // Launches under one round ask for two slots for each of up to 8 workgroups per task, at most one per compute unit,
    // as the planning test pins it; the parts need no more than that (2 cut < 2 cus slots, or cut * shares <= cus of them
    // and 32 bytes per task).
    plan->room = whole > 0 && !always ? plan->bytes()
                                      : (((size_t)tasks * 4 + 255) & ~(size_t)255) +
                                            2 * (size_t)std::min<int64_t>(cus, tasks * kSdpaSplitNodes) * slot;
  }
  return true;
}

static bool sdpa_premul(const SdpaArgs& a) { return !(a.scale_log2e > 0.f && a.scale_log2e < 1e30f); }
// one K and one V segment whose rows lie within 2 GiB of the head's first row: 32-bit offsets
static bool sdpa_oneseg(const SdpaArgs& a) {
  return a.n_kvseg == 1 && a.k[0].ss > 0 && a.v[0].ss > 0 && a.Skv < (1 << 30) && (a.Skv + 2 * BKV) * a.k[0].ss * 2 < 0x7fffffffLL &&
         (a.Skv + 2 * BKV) * a.v[0].ss * 2 < 0x7fffffffLL;
}

template <int DP, int DL, bool M16, int KG>
static dt_status launch(hipStream_t s, SdpaArgs a) {
  a.q_norm = 0;
  a.q_aligned = (reinterpret_cast<uintptr_t>(a.q_rot) & 15) == 0;
  for (int i = 0; i < a.n_qseg; i++) {
    a.q_norm |= a.q_gamma[i] != nullptr;
    a.q_aligned &= (reinterpret_cast<uintptr_t>(a.q_gamma[i]) & 15) == 0;
  }
  a.q_tiles = (int)((a.Sq + query_rows(KG) - 1) / query_rows(KG));
  int64_t total = (int64_t)a.q_tiles * a.Hq * a.B;
  if (total > 0x7fffffff) return DT_NO_KERNEL;
  a.total_blocks = (int)total;
  const bool premul = sdpa_premul(a), oneseg = sdpa_oneseg(a);
  dim3 block(512);
  dim3 grid((unsigned)total);
  if constexpr (KG == 1) {
    if (a.partials) {
      // key-split launch: the counters start at zero
      if (!a.counters_zeroed) {
        const int n = a.cut_tasks * kSdpaSplitNodes;
        hipLaunchKernelGGL(sdpa_zero_counters_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, a.counters, n);
        if (const dt_status st = launch_status(); st != DT_OK) return st;
      }
      a.total_blocks = a.cut_tasks * a.shares;  // (of the cut tasks)
      grid = dim3((unsigned)(a.whole_tasks + a.total_blocks));
      if (oneseg) {
        if (premul) hipLaunchKernelGGL((sdpa_kernel<DP, DL, M16, true, true, true, 1>), grid, block, 0, s, a);
        else hipLaunchKernelGGL((sdpa_kernel<DP, DL, M16, false, true, true, 1>), grid, block, 0, s, a);
      } else {
        if (premul) hipLaunchKernelGGL((sdpa_kernel<DP, DL, M16, true, false, true, 1>), grid, block, 0, s, a);
        else hipLaunchKernelGGL((sdpa_kernel<DP, DL, M16, false, false, true, 1>), grid, block, 0, s, a);
      }
      return launch_status();
    }
    if (premul) {
      if (oneseg) hipLaunchKernelGGL((sdpa_kernel<DP, DL, M16, true, true, false, 1>), grid, block, 0, s, a);
      else hipLaunchKernelGGL((sdpa_kernel<DP, DL, M16, true, false, false, 1>), grid, block, 0, s, a);
      return launch_status();
    }
  }
  if (oneseg) hipLaunchKernelGGL((sdpa_kernel<DP, DL, M16, false, true, false, KG>), grid, block, 0, s, a);
  else hipLaunchKernelGGL((sdpa_kernel<DP, DL, M16, false, false, false, KG>), grid, block, 0, s, a);
  return launch_status();
}

// Estimated time (us) of a launch: `launch` once, and for every round of workgroups `round` and its steps, each of a key tile a
// key group, which take `few` where few compute units are at work and `all` where all of them are.  Fits to 1000 launches of 256 ..
// 5000 queries and 64 .. 5000 keys in two segments, 4 .. 24 heads, on the whole card: half of them within 4 %, nineteen of twenty within 12 %.
// (Keys in one segment are 3 .. 10 % faster in either form; which form is taken does not depend on it, since results may not.)
struct SdpaRate {
  double few, all, round, launch;
  double rounds(int64_t workgroups, int64_t steps, int cus) const {
    const int64_t full = workgroups / cus, rest = workgroups % cus;
    return (double)full * ((double)steps * all + round) + (rest ? (double)steps * (few + (all - few) * (double)rest / cus) + round : 0.0);
  }
};
// head sizes up to 48 (whose kernels were some 3 % faster then, in either form), 64, 80, 128
constexpr SdpaRate kOneGroup[4] = {{1.027, 1.087, 4.95, 1.946}, {1.02, 1.135, 6.472, 1.362}, {1.372, 1.511, 7.612, 1.745}, {1.326, 1.718, 9.237, 1.29}};
constexpr SdpaRate kTwoGroups[4] = {{1.217, 1.244, 5.799, 2.19}, {1.279, 1.273, 6.058, 2.126}, {1.78, 1.844, 8.872, 1.35}, {1.662, 2.053, 9.644, 2.347}};

// Whether a launch runs with two key groups to a workgroup.  Its tasks then are half as large, which fills the compute units where there
// are few of them and wastes less of a last round: us, one group / two, head size 128, 12 x 1050 x 1050 30.8 / 23.8, 10 x 2472 x 2472 63.9 /
// 43.8, 24 x 2637 x 2637 (in place of a cut last round) 109 / 93, 20 x 3160 x 545 43.3 / 36.4; 40 and 64, 4 x 1582 x 1582 26.7 / 20.1, 24 x 2637
// x 2637 74 / 58.  But every key tile is fetched for half as many queries, and rounds of full-length tasks are slower: 40 x 8000 x 8000 1077 /
// 1236, 24 x 4608 x 4608 232 / 290.  Taken where the estimate gains 3 %: 0.87 .. 0.92 of the time, by head size and segments, of 2000 random launches,
// the worst of which takes 1.03.
static bool sdpa_two_groups(const SdpaArgs& a) {
  const char* knob = getenv("DT_SDPA_KEY_SPLIT");  // "groups": wherever it can be; "never" and "always" (sdpa_split_plan): no
  if (knob && (knob[0] == 'n' || knob[0] == 'a' || knob[0] == 'g')) return knob[0] == 'g';
  // a launch that was to be cut and got no workspace for it keeps the whole tasks that such calls have always had
  if (!a.partials && sdpa_split_plan(a.B, a.Hq, a.D, a.Sq, a.Skv, nullptr)) return false;
  const int size = a.D <= 48 ? 0 : a.D <= 64 ? 1 : a.D <= 80 ? 2 : 3;
  const SdpaRate &one = kOneGroup[size], &two = kTwoGroups[size];
  const int cus = compute_units();
  const int64_t heads = (int64_t)a.B * a.Hq, n_tiles = (a.Skv + BKV - 1) / BKV;
  const auto tasks = [&](int kg) { return heads * ((a.Sq + query_rows(kg) - 1) / query_rows(kg)); };
  double t1 = one.launch;
  if (a.partials) {  // (a cut costs another 16 us, 10 at head sizes up to 64)
    const int64_t parts = (int64_t)a.cut_tasks * a.shares;
    t1 += one.rounds(a.whole_tasks, n_tiles, cus) + one.rounds(parts, (n_tiles + a.shares - 1) / a.shares, cus) + (a.D <= 64 ? 10.0 : 16.0);
  } else {
    t1 += one.rounds(tasks(1), n_tiles, cus);
  }
  return two.launch + two.rounds(tasks(2), (n_tiles + 1) / 2, cus) < 0.97 * t1;
}

dt_status sdpa_launch(hipStream_t s, const SdpaArgs& a) {
  if (a.B <= 0 || a.Sq <= 0) return DT_OK;
  // Head sizes up to 64 have an exponential for every two to four MFMAs and are bound by the exponentials (M16: 4096 queries,
  // 16 heads of 40 73 us against 81, 20 heads of 64 113 against 122).  Above, 16x16x32 is ahead where the workgroups fill
  // the card, whose power then is the limit, and behind where under seven tenths of the compute units have one and the clock
  // stays up (us, 32x32x16 / 16x16x32, head size 128: 120 workgroups 34.8 / 36.9, 144 101 / 108, 168 47.2 / 48.3, 192 104
  // / 99, 216 66.9 / 63.1, 432 250 / 235 alone in a loop and 258 / 255 behind a block's projections, 1440 of 141 key tiles 1495 /
  // 1398; head size 80: 144 56.7 / 58.4, 256 113 / 96).
  // Cut along the keys, launches of up to one round are limited by power only where the parts are many and long: 16x16x32 takes
  // 1.06 times as long with under 100 of them and 1.02 .. 1.03 with 220 .. 256 of up to 8 key tiles; from 200 parts of 16 key
  // tiles on it takes 1.00 .. 0.97, behind whole rounds 0.97 (means of 1400 launches of head sizes 88 .. 128; us, 12 heads of 128, 323 x
  // 1928 34.2 / 35.9, 4 heads, 4096 x 4096 60.3 / 58.0, 264 tasks 111 / 109).
  // Head sizes up to 80 multiply 80 columns in this form only, which decides for it wherever the launch is cut (0.83 .. 0.98).
  // (a scale that is folded into the scores first has one key group)
  if (!sdpa_premul(a) && sdpa_two_groups(a)) {
    SdpaArgs u = a;
    u.partials = nullptr;  // uncut, whatever the workspace
    if (a.D <= 48) return launch<64, 48, false, 2>(s, u);
    if (a.D <= 64) return launch<64, 64, false, 2>(s, u);
    if (a.D <= 80) return launch<128, 80, true, 2>(s, u);
    return launch<128, 128, false, 2>(s, u);  // (16x16x32 is 0 .. 7 % slower here, in launches of one round and of many)
  }
  if (a.D <= 64) return launch<64, 64, false, 1>(s, a);
  const int64_t tasks = (a.Sq + query_rows(1) - 1) / query_rows(1) * a.Hq * a.B;
  const int64_t cus = compute_units();
  const auto short_parts = [&] { return (int64_t)a.cut_tasks * a.shares * 10 < cus * 8 || (a.Skv + BKV - 1) / BKV < 16 * a.shares; };
  if (a.partials ? a.D > 80 && a.whole_tasks == 0 && short_parts() : tasks * 10 < cus * 7) return launch<128, 128, false, 1>(s, a);
  if (a.D <= 80) return launch<128, 80, true, 1>(s, a);
  return launch<128, 128, true, 1>(s, a);
}

}  // namespace dt
