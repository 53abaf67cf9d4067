// K1: Dense over palettized weights, Y = X W^T (+ bias), for gfx950.
//
// The tiled kernel takes weights packed: per K-tile two threads
// per weight row each pull half of a 32-index granule into registers, unpack
// it, look the fp16 values up in palettes held in LDS, and write the fp16 row
// slice into an LDS ring that v_mfma_f32_16x16x32_f16 then consumes; X (and a
// plain fp16 weight) goes from memory straight into LDS.  Where many rows of X
// would have it look every weight up once per tile of rows, and the caller has
// scratch for them, fp16 copies of the weights are written first and the launch
// runs on those (plan_copies).  fp32 accumulation,
// one rounding to fp16, optional fused tails (per-head RMSNorm + RoPE, or
// activation / gate / fp32 residual).
//
// Tile: BM x BN outputs per 512-thread workgroup (8 waves, two per SIMD, each
// a BN/2 x BM/4 slice), K-tiles of 32 processed in pairs; one barrier per K-tile
// (per pair with plain fp16 weights, which no wave writes to LDS itself).  Transfers
// from memory are waited for once per K-tile, on the 128 x 128 tile with
// palettes in LDS and with plain fp16 weights once per pair.
#include <algorithm>
#include <cmath>
#include <cstdlib>

#include "dt_dense_any.h"
#include "dt_dense_launch.h"
#include "dt_dense_rows.h"
#include "dt_depalettize.h"
#include "dt_lora.h"

namespace dt {

extern template dt_status launch_dense_q<4>(hipStream_t, const DenseArgs&, int, bool, int);
extern template dt_status launch_dense_q<5>(hipStream_t, const DenseArgs&, int, bool, int);
extern template dt_status launch_dense_q<6>(hipStream_t, const DenseArgs&, int, bool, int);
extern template dt_status launch_dense_q<7>(hipStream_t, const DenseArgs&, int, bool, int);
extern template dt_status launch_dense_q<8>(hipStream_t, const DenseArgs&, int, bool, int);
extern template dt_status launch_dense_q<16>(hipStream_t, const DenseArgs&, int, bool, int);

// the kernel with the elementwise tail only when some weight of the launch asks for one
static dt_status launch_dense(hipStream_t s, const DenseArgs& a, int tile, int qbits, int mode) {
  bool post = false;
  for (int i = 0; i < kMaxWeights; i++) post = post || a.w[i].act != DT_ACT_NONE || a.w[i].gate || a.w[i].res || a.w[i].add || a.w[i].mul || a.w[i].scale != 1.0f;
  switch (qbits) {
    case 4: return launch_dense_q<4>(s, a, tile, post, mode);
    case 5: return launch_dense_q<5>(s, a, tile, post, mode);
    case 6: return launch_dense_q<6>(s, a, tile, post, mode);
    case 7: return launch_dense_q<7>(s, a, tile, post, mode);
    case 8: return launch_dense_q<8>(s, a, tile, post, mode);
    case 16: return launch_dense_q<16>(s, a, tile, post, mode);
  }
  return DT_INVALID;
}

constexpr int kDenseCUs = 256;  // compute units of the whole card

// K-tiles from one at which rows may enter new blocks to the next.
static int64_t pal_step(int64_t K, int nib) { return std::gcd(K, (int64_t)nib) / BK; }

// Palette placement for a BN-row tile (see PalMode) in a launch of `tiles` of them (0: of more than the compute units).
static int choose_pal_mode(int qbits, int nib, int64_t K, int BM, int BN, int64_t tiles = 0) {
  if (qbits == 16) return kPlainF16;
  const int64_t pal_bytes = (int64_t)2 << qbits;
  const int64_t shared_count = ((int64_t)BN * K) / nib + 2;
  const bool row = (int64_t)BN * pal_bytes <= pal_lds_bytes(BM, BN, kPalRow);
  const bool shared = !(BM == 256 && BN == 128) && shared_count * pal_bytes <= pal_lds_bytes(BM, BN, kPalShared);
  // a per-row table has no bank conflicts, but 128- and 256-entry palettes make one of 32 or 64 KB: the 128 x 128 tile
  // takes it where the palettes of its blocks would not fit the 24 KB that let two workgroups share a compute unit, and
  // where there is none to share with and rows enter new blocks at every 16th K-tile at most (us, shared / per row, 250
  // tiles: q7p K = 1024 27.5 / 25.2, 1536 37.7 / 35.2, 2048 48.5 / 42.1, 4096 89.0 / 76.5; q8p 27.2 / 25.6, 37.3 / 37.0,
  // 47.6 / 42.7, 87.5 / 76.0; at every 8th, K = 1792, q7p 43.2 / 42.9, q8p 42.7 / 46.4; 512 tiles, which do share, K = 2048
  // q8p 62.9 / 80.4)
  const bool small = BM == 128 && BN == 128;
  const int64_t step = pal_step(K, nib);
  if (shared && small && qbits >= 7 && (tiles == 0 || tiles > kDenseCUs || step < 16)) return kPalShared;
  // And where some row may enter a new block at every second K-tile (K an odd multiple of 64), that check, its barrier
  // and the 64 entries to rewrite cost more than conflicts do (us, per row / shared: 8192 x 320 -> 960 19.1 / 17.7,
  // 4608 x 960 -> 3072 48.0 / 42.8, 2048 x 1344 -> 4096 51.5 / 43.8, on 128 x 128 tiles 2016 x 1600 -> 1280 42.6 / 35.8);
  // at every fourth they are even on the small tile (4096 x 640 -> 640 17.9 / 17.5), at every eighth the table is
  // ahead (2016 x 1280 -> 1280 28.2 / 29.8).  Palettes of 16 and 32 entries are rewritten fast enough (4096 x 320 ->
  // 1280: q5p 16.5 / 16.4, q4p 16.2 / 16.4).
  if (shared && qbits == 6 && (small ? step <= 4 : BN == 256 && step <= 2)) return kPalShared;
  if (row) return kPalRow;
  if (shared) return kPalShared;
  return kPalGlobal;
}

}  // namespace dt

namespace dt {

// One Dense problem as the entry points receive it.
struct HostGroup {
  int64_t M, K;
  const uint16_t* X;
  int64_t ldx;
  const dt_qx_weight* W;
  int32_t n_weights;
  const uint16_t* const* bias;
  uint16_t* const* Y;
  const int64_t* ldy;
  const dt_head_epilogue* epi;
  const dt_dense_post* post;

  bool wants_epi(int wi) const { return epi && (epi[wi].gamma || epi[wi].rot); }
  // fused head epilogue: in the tiled kernel for 128-wide heads that start on a 16-byte aligned,
  // 8-element-strided output; otherwise the Dense runs plain and the norm / rotation pass follows
  bool fusable(int wi) const {
    return epi[wi].head_dim == 128 && (ldy[wi] % 8 == 0) && ((reinterpret_cast<uintptr_t>(Y[wi]) & 15) == 0) &&
           (!epi[wi].gamma || (reinterpret_cast<uintptr_t>(epi[wi].gamma) & 7) == 0) &&
           (!epi[wi].rot || (reinterpret_cast<uintptr_t>(epi[wi].rot) & 7) == 0) &&
           (!bias || !bias[wi] || (reinterpret_cast<uintptr_t>(bias[wi]) & 7) == 0);
  }
  // (the tiled kernel addresses X and the packed weight with 32-bit byte offsets from their bases)
  bool x_ok() const {
    return (K % (2 * BK) == 0) && (ldx % 8 == 0) && ((reinterpret_cast<uintptr_t>(X) & 15) == 0) &&
           (M == 0 || ((M - 1) * ldx + K) * 2 <= (int64_t)0xffffffff);
  }
  bool w_tiled(int wi) const {
    const dt_qx_weight& w = W[wi];
    if (!(w.count / K > 0 && (reinterpret_cast<uintptr_t>(w.data) & 15) == 0 && (w.qbits == 16 || w.nib % 32 == 0))) return false;
    const int64_t bytes = w.qbits == 16 ? w.count * 2 : dt_qx_bytes(w.qbits, w.nib, w.count);
    return bytes > 0 && bytes <= (int64_t)0xffffffff;
  }
};

static dt_status validate_group(const HostGroup& h) {
  if (h.epi && h.n_weights > 0) {
    for (int i = 0; i < h.n_weights; i++) {
      const dt_head_epilogue& e = h.epi[i];
      if (!e.gamma && !e.rot) continue;
      if (e.head_dim <= 0 || e.head_dim % 2 != 0 || e.head_dim > 128) return DT_NO_KERNEL;
      if (e.rot && e.rot_pos0 < 0) return DT_INVALID;
      if (h.Y && h.ldy && h.M > 0 && ((h.ldy[i] & 1) || (reinterpret_cast<uintptr_t>(h.Y[i]) & 3))) return DT_INVALID;
      if (e.rot && (reinterpret_cast<uintptr_t>(e.rot) & 3)) return DT_INVALID;
      if (h.W && h.K > 0 && h.W[i].count >= 0 && (h.W[i].count / h.K) % e.head_dim != 0) return DT_INVALID;
    }
  }
  if (h.M < 0 || h.K <= 0 || h.n_weights <= 0 || !h.W || !h.Y || !h.ldy) return DT_INVALID;
  if (h.post && h.epi) return DT_INVALID;
  if (h.post)
    for (int i = 0; i < h.n_weights; i++) {
      const dt_dense_post& p = h.post[i];
      if (p.activation < DT_ACT_NONE || p.activation > DT_ACT_GELU_ERF) return DT_INVALID;
      if (p.multiplicand && ((reinterpret_cast<uintptr_t>(p.multiplicand) & 1) || (h.W && h.K > 0 && p.ld_multiplicand < h.W[i].count / h.K)))
        return DT_INVALID;
      if (p.residual && ((reinterpret_cast<uintptr_t>(p.residual) & 3) || (h.W && h.K > 0 && p.ld_residual < h.W[i].count / h.K)))
        return DT_INVALID;
      if (p.addend && ((reinterpret_cast<uintptr_t>(p.addend) & 1) || (h.W && h.K > 0 && p.ld_addend < h.W[i].count / h.K)))
        return DT_INVALID;
      if (!(p.scale == p.scale) || p.scale - p.scale != 0.f) return DT_INVALID;  // NaN or infinite
      if (p.gate_f32 && (!p.residual || p.gate || (reinterpret_cast<uintptr_t>(p.gate_f32) & 3))) return DT_INVALID;
    }
  if (h.M > 0x7fffffff || h.K > 0x7fffffff) return DT_INVALID;
  for (int i = 0; i < h.n_weights; i++) {
    const dt_qx_weight& w = h.W[i];
    if (!w.data || w.count < 0 || w.count % h.K != 0) return DT_INVALID;
    if (w.qbits != 16 && (w.qbits < 4 || w.qbits > 8 || w.nib <= 0)) return DT_INVALID;
    if (w.count / h.K > 0x7fffffff) return DT_INVALID;
    const bool to_residual_only = h.post && h.post[i].residual && !h.Y[i];
    if (h.M > 0 && !to_residual_only && (!h.Y[i] || h.ldy[i] < w.count / h.K)) return DT_INVALID;
  }
  if (h.M > 0 && (!h.X || h.ldx < h.K)) return DT_INVALID;
  return DT_OK;
}

static dt_status epilogue_pass(hipStream_t s, const HostGroup& h, int wi) {
  QkPrepArgs p;
  p.src = h.Y[wi];
  p.dst = h.Y[wi];
  p.src_sb = p.dst_sb = 0;
  p.src_ss = p.dst_ss = h.ldy[wi];
  p.src_sh = p.dst_sh = h.epi[wi].head_dim;
  p.B = 1;
  p.S = h.M;
  p.H = (int32_t)((h.W[wi].count / h.K) / h.epi[wi].head_dim);
  p.D = h.epi[wi].head_dim;
  p.gamma = h.epi[wi].gamma;
  p.eps = h.epi[wi].eps;
  p.norm_per_head = 1;
  p.rot = h.epi[wi].rot;
  p.rot_pos0 = h.epi[wi].rot_pos0;
  p.post_scale = 1.0f;
  return qk_prep_launch(s, p);
}

// dt_dense_post::scale as the kernels take it: 0 (a zeroed struct) means none.
static float post_scale(const HostGroup& h, int wi) {
  return h.post && h.post[wi].scale != 0.f ? h.post[wi].scale : 1.0f;
}

// Appends weight wi of h to the launch; returns its number of N-tiles.
static int add_weight(DenseArgs& a, int slot, const HostGroup& h, int wi, int tile_begin, int BN, bool fuse) {
  const int64_t n_rows = h.W[wi].count / h.K;
  DenseWeight& d = a.w[slot];
  d.data = static_cast<const uint8_t*>(h.W[wi].data);
  d.bias = h.bias ? h.bias[wi] : nullptr;
  d.y = h.Y[wi];
  d.ldy = h.ldy[wi];
  d.n = (int32_t)n_rows;
  d.tile_begin = tile_begin;
  d.gamma = fuse ? h.epi[wi].gamma : nullptr;
  d.rot = fuse ? h.epi[wi].rot : nullptr;
  d.rot_pos0 = fuse ? h.epi[wi].rot_pos0 : 0;
  d.eps = fuse ? h.epi[wi].eps : 0.f;
  d.scale = post_scale(h, wi);
  d.add = h.post ? h.post[wi].addend : nullptr;
  d.ld_add = h.post ? h.post[wi].ld_addend : 0;
  d.act = h.post ? h.post[wi].activation : DT_ACT_NONE;
  d.gate = h.post ? h.post[wi].gate : nullptr;
  d.res = h.post ? h.post[wi].residual : nullptr;
  d.ld_res = h.post ? h.post[wi].ld_residual : 0;
  d.gate32 = h.post ? h.post[wi].gate_f32 : nullptr;
  d.mul = h.post ? h.post[wi].multiplicand : nullptr;
  d.ld_mul = h.post ? h.post[wi].ld_multiplicand : 0;
  return (int)((n_rows + BN - 1) / BN);
}

static void finish_args(DenseArgs& a, int n_groups, int n_w, int64_t K, const dt_qx_weight& w0) {
  for (int j = n_w; j < kMaxWeights; j++) a.w[j] = a.w[0];
  for (int j = n_groups; j < kMaxGroups; j++) a.g[j] = a.g[0];
  a.n_groups = n_groups;
  a.lora = DenseLora{};
  a.k = (int32_t)K;
  a.nib = w0.qbits == 16 ? 32 : w0.nib;
  a.pal_step = (int32_t)pal_step(K, a.nib);
}

// How a launch of the tiled kernel is laid out: its tile and, where the tiles do not fill the compute units evenly, how
// many of them are cut along K into how many shares.
struct TilePlan {
  int tile = kTile256x256, BM = 256, BN = 256;
  int64_t tiles = 0;
  int64_t whole = 0;  // tiles that stay whole; the rest is cut into `split` shares each
  int split = 1;
  bool act = false;  // some weight's tail has an activation
  int64_t x_bytes = 0;  // of all problems' rows
  size_t expand_bytes = 0;  // > 0: the weights are written out as fp16 in front of the launch, to this much scratch
  int expanded = 0;         // that many of them
  // workspace of the split tiles: their counters, then their slots
  size_t counter_bytes() const { return split > 1 ? ((size_t)(tiles - whole) * kSplitNodes * 4 + 255) & ~(size_t)255 : 0; }
  size_t split_bytes() const { return split > 1 ? counter_bytes() + (size_t)((tiles - whole) * split * dense_split_slot_bytes(BM, BN)) : 0; }
  size_t bytes() const { return expand_bytes + split_bytes(); }
};

// Fewer 256 x 256 tiles than this leave too many of the 256 compute units idle: such launches take 128 x 128 tiles.
constexpr int64_t kFillTiles = 192;
constexpr size_t kDenseMaxWorkspace = (size_t)128 << 20;
// fp16 copies of a launch's weights.  Over 200 MiB they leave the memory-side cache (256 MB) before the launch has read them,
// which launches of few rows, that wait for the weights, do not make up for (us, packed / copied: 373 x 10368 -> 2 x 6144 q5p, 255
// MB, 180 / 218; 353 x 8832 -> 12352 q6p, 218 MB, 167 / 186; 468 x 12416 -> 2 x 5248 q8p, 261 MB, 243 / 289; below the line 512
// x 5120 -> 5120 q6p, 52 MB, 71 / 52; 300 x 5120 -> 5120 q8p 56 / 49; 568 x 7488 -> 11648 q6p, 174 MB, 250 / 149).
constexpr size_t kDenseMaxExpand = (size_t)512 << 20;
constexpr size_t kDenseFewRowsExpand = (size_t)200 << 20;
constexpr int64_t kDenseFewRows = 640;
constexpr int64_t kDenseNearX = (int64_t)48 << 20;

// Estimated time (us) of a launch whose rows enter new blocks at every `step`-th K-tile at most: a fit to 930 launches of
// 65 .. 4000 rows on the whole card (part of one would need costs of its own; the results do not depend on the layout
// chosen beyond the order of the sums), made on kernels with 32x32x16 instructions, nine tenths of them within a tenth then.  Against the
// present ones (8100 launches of 65 .. 8192 rows of random sizes, replayed from graphs) it is high for uncut 128 x 128 tiles,
// 1.29 times the measured time with packed weights and 1.41 with plain ones (medians; they take some 4 us less than the 7.7 outside the
// K loop), and 0.94 .. 1.15 on the other shapes and on cuts.  The choice between packed weights and copies, which takes 0.93 of it for
// these, falls on the slower by 5 % and 3 us in 346 of 6154 launches, 1.4 % of the time of all.  Priced are: one workgroup's K-tile on each
// tile shape, the cheaper the more compute units idle (the card is limited as a whole); what entering new blocks adds to it
// where every row has a table of its own to rewrite, most for 128 and 256 entries; the time outside the K loop; two
// 128 x 128 tiles that share a compute unit, except with per-row tables of 32 or 64 KB beside the other 56, which take it in
// turns; and cutting: the launch that zeroes the counters and, for each level of meetings, a way out and in for the sums.
// (us, uncut / cut: 512 x 5120 -> 2 x 5120 q5p 117 / 88, 128 x 5120 -> 1152 q8p 90 / 37; and left whole because of these
// terms: 3 x (571 x 4288 -> 7872) q7p 251 / 342, 1000 x 1792 -> 4096 q7p 42 / 48, 721 x 7168 -> 2560 fp16 46 / 52.)
// `expanded`: plain weights that a launch of their own writes first, which also zeroes the counters.
static double plan_cost(const TilePlan& p, int qbits, int mode, int nk, int64_t step, bool expanded) {
  const bool plain = qbits == 16, wide = qbits == 7 || qbits == 8, row = mode == kPalRow;
  const double entering = row ? (wide ? 0.70 : 0.33) / (double)step : 0.0;
  // An X so large that it has left the memory-side cache when the copies behind it are written: a workgroup that has a compute unit to
  // itself and two K-tiles on their way waits for memory, however few of them there are.  (us, 12288 -> 3072 in Flux blocks, 192 x 256 /
  // 256 x 256 / 128 x 256 cut: 2577 rows 265 / 297 / 190, 2777 274 / 296 / 244, 3377 284 / 304 / 265, 3677 283 / 310 / 291, 4608 382 / 313 / 349; by itself,
  // with X in the cache, 3112 rows 212 / 222 / 220.)
  const bool far = plain && expanded && p.x_bytes > kDenseNearX;
  // one workgroup's K-tile with the share `busy` of the compute units at work
  const auto k_tile = [&](double busy) -> double {
    switch (p.tile) {
      case kTile256x256: return far ? 0.66 + 0.15 * busy : plain ? 0.37 + 0.44 * busy : (wide ? 0.71 + 0.47 * busy : 0.73 + 0.27 * busy) + entering;
      case kTile192x256: return far ? 0.58 + 0.13 * busy : 0.30 + 0.30 * busy;
      case kTile128x256: return plain ? 0.28 + 0.14 * busy : wide ? 0.85 + 0.10 * busy : (row ? 0.60 : 0.78) + 0.17 * busy + entering;
      case kTile128x128: return plain ? 0.145 + 0.09 * busy : row ? 0.49 + 0.06 * busy + entering : wide ? 0.575 + 0.065 * busy : 0.56 + 0.09 * busy;
    }
    return 0.51 + 0.195 * busy + entering;
  };
  double outside = p.tile == kTile256x256 ? 11.3 : p.tile == kTile192x256 ? 12.3 : p.tile == kTile128x128 ? 7.7 : 7.1;
  // an activation's arithmetic (us, none / GELU, plain weights: one round of 256 x 256 tiles 33.4 / 42.4 and 48.6 / 56.7, of 192 x 256 45.9 / 51.2
  // and 94.4 / 97.6; 2.5 rounds of 128 x 256 33.8 / 45.9, of two 128 x 128 a compute unit 26.9 / 34.8)
  if (p.act) outside += p.tile == kTile256x256 ? 9.0 : p.tile == kTile192x256 ? 5.0 : p.tile == kTile128x128 ? 3.3 : 4.5;
  const bool pairs_of_tiles = p.tile == kTile128x128 && !(row && wide);
  // `n` workgroups of `kt` K-tiles each
  const auto time = [&](int64_t n, int kt) -> double {
    if (n == 0) return 0.0;
    if (pairs_of_tiles && n > kDenseCUs) {
      const double both = (plain ? 0.54 : wide ? 0.97 : 0.90) + entering, gap = plain ? 0.095 : wide ? 0.24 : 0.20;
      const int64_t full = n / (2 * kDenseCUs), rest = n % (2 * kDenseCUs);
      const double last = both * (double)rest / (2 * kDenseCUs);
      if (full == 0) return std::max(k_tile(1.0) + gap, last) * kt + outside;
      return ((double)full * both + (rest ? std::max(0.35 * both, last) : 0.0)) * kt + outside * (double)(full + (rest ? 1 : 0));
    }
    const int64_t full = n / kDenseCUs, rest = n % kDenseCUs;
    return (double)full * (kt * k_tile(1.0) + outside) + (rest ? kt * k_tile((double)rest / kDenseCUs) + outside : 0.0);
  };
  if (p.split == 1) return time(p.tiles, nk);
  const int64_t shares = (p.tiles - p.whole) * p.split;
  const int levels = p.split > 4 ? 3 : p.split > 2 ? 2 : 1;
  const double mb = 1e-6 * (double)(shares * dense_split_slot_bytes(p.BM, p.BN));
  return time(p.whole, nk) + time(shares, 2 * ((nk / 2 + p.split - 1) / p.split)) + (expanded ? 0.0 : 5.0) + levels * (3.5 + 0.095 * mb);
}

// The best way to cut tiles of `base`'s shape that `ws_bytes` of workspace allow: all of them, or those of the last,
// unfilled round of workgroups.  None of up to 32 K-tiles (K = 1024): a cut would gain a few us of 25 at most.
static TilePlan best_split(const TilePlan& base, int qbits, int mode, int nk, int64_t step, bool expanded, size_t ws_bytes,
                            double* cost) {
  TilePlan best = base;
  best.split = 1;
  best.whole = base.tiles;
  *cost = plan_cost(best, qbits, mode, nk, step, expanded);
  for (int s = 2; nk > 32 && s <= kMaxSplit && nk / s >= 8; s++)
    for (const int64_t whole : {(int64_t)0, base.tiles / kDenseCUs * kDenseCUs}) {
      TilePlan p = base;
      p.split = s;
      p.whole = whole;
      if (p.whole >= p.tiles || p.bytes() > ws_bytes || p.bytes() > kDenseMaxWorkspace) continue;
      const double t = plan_cost(p, qbits, mode, nk, step, expanded);
      if (t < (best.split > 1 ? 0.97 : 1.0) * *cost) {  // (a finer cut, of more memory, has to be worth it)
        *cost = t;
        best = p;
      }
    }
  return best;
}

// The layout of one launch over problems hs[0 .. n) (weights [w_begin, w_end) of each; they share K and the weight
// format, which w0 stands for; `expanded`: plain fp16, as the copies of palettized weights are).  `wide`: a fused head
// epilogue needs tiles of 256 features.  *cost: its estimate.
static TilePlan plan_format(const HostGroup* hs, int n, int w_begin, int w_end, bool wide, size_t ws_bytes,
                            const dt_qx_weight& w0, bool expanded, double* cost) {
  const int64_t K = hs[0].K;
  const int nk = (int)(K / BK);
  const auto shape = [&](int tile, int BM, int BN) {
    TilePlan p;
    p.tile = tile;
    p.BM = BM;
    p.BN = BN;
    for (int gi = 0; gi < n; gi++) {
      p.x_bytes += 2 * hs[gi].M * K;
      for (int j = w_begin; j < (n > 1 ? hs[gi].n_weights : w_end); j++) {
        p.act = p.act || (hs[gi].post && hs[gi].post[j].activation != DT_ACT_NONE);
        p.tiles += ((hs[gi].M + BM - 1) / BM) * ((hs[gi].W[j].count / K + BN - 1) / BN);
      }
    }
    p.whole = p.tiles;
    return p;
  };
  int64_t m_max = 0, n_max = 0;
  for (int gi = 0; gi < n; gi++) {
    m_max = std::max(m_max, hs[gi].M);
    n_max = std::max(n_max, hs[gi].W[w_begin].count / K);
  }
  // (palettes that fit beside no big tile -- 256-entry palettes with small blocks -- would be looked up in memory:
  // the small tile holds a per-row table of them and is several times faster, unless a fused epilogue needs the big one)
  const bool pal_fits_big = choose_pal_mode(w0.qbits, w0.nib, K, 256, 256) != kPalGlobal ||
                            choose_pal_mode(w0.qbits, w0.nib, K, 128, 128) == kPalGlobal;
  const TilePlan t256 = shape(kTile256x256, 256, 256), tnarrow = shape(kTile128x256, 128, 256);
  const TilePlan ttall = shape(kTile256x128, 256, 128), tsmall = shape(kTile128x128, 128, 128);
  const bool tall_ok = (w0.qbits == 7 || w0.qbits == 8) && choose_pal_mode(w0.qbits, w0.nib, K, 256, 128) == kPalRow;
  // (plain fp16 weights with one or two pairs of K-tiles -- a LoRA's up projection -- are all prologue and output, which two
  // small tiles on a compute unit hide for each other: us, 256 x 256 / 128 x 128, 4608 x 64 -> 3072 with an addend 22.9 /
  // 21.0, -> 12288 81.5 / 66.7, 1900 x 128 -> 9216 25.3 / 19.3; 8192 x 64 -> 2048 14.9 / 14.7)
  const bool brief = w0.qbits == 16 && K <= 128;
  const bool big = (((m_max >= 1024) && (n_max >= 256) && t256.tiles >= kFillTiles) && pal_fits_big && !brief) || wide;
  TilePlan base = big ? (m_max < 1024 ? tnarrow : t256) : (!pal_fits_big && tall_ok && m_max >= 1024 && n_max >= 128 && t256.tiles * 2 >= kFillTiles) ? ttall : tsmall;
  const auto pal_mode = [&](const TilePlan& p) { return choose_pal_mode(w0.qbits, w0.qbits == 16 ? 32 : w0.nib, K, p.BM, p.BN, p.tiles); };
  const int64_t step = pal_step(K, w0.qbits == 16 ? 32 : w0.nib);
  double start = plan_cost(base, w0.qbits, pal_mode(base), nk, step, expanded);
  // Plain weights: tiles of 192 tokens where the rounds of the others come out badly filled, and under an activation, which big tiles do with
  // nothing beside it on the compute unit, small ones, whose estimate is high.  The sums are the same on every tile.  us, without
  // / with these, of 130 launches of random sizes the slowest by 3 % and half of them faster by 3 % and more: 1 x (2304 x 2048 -> 5120) fp16 57.2 / 45.9
  // (240 tiles, 720 of 128 x 128), 3394 x 4544 -> 3200 q8p 115.8 / 97.2, 4108 x 2048 -> 2816 q8p 64.9 / 53.3, 2 x (576 x 2368 -> 10368) q6p 128.9 /
  // 77.0, with GELU 2016 x 1280 -> 5120 fp16 44.2 / 38.2, 2 x (4531 x 448 -> 5888) q6p 121.1 / 102.7, 3 x (5454 x 320 -> 960) q8p 54.2 / 39.1, 1376 x 3072 -> 12288
  // 134 on 288 tiles of 256 x 256, 117 cut, 112 on 384 of these; left as it was: 3500 x 1280 -> 3840 fp16 36.6 on 210 tiles of 256 x 256, 54.6 on 285.
  if (w0.qbits == 16 && !brief) {
    const auto instead = [&](const TilePlan& p, double factor) {
      const double t = factor * plan_cost(p, 16, kPlainF16, nk, step, expanded);
      if (t < 0.95 * start) {
        start = t;
        base = p;
      }
    };
    if (m_max > 128 && n_max >= 256) instead(shape(kTile192x256, 192, 256), 1.0);
    if (base.act && !wide && base.tile != kTile128x128) instead(tsmall, 1.0 / 1.15);
  }
  *cost = start;
  // Without workspace the rules above stand.  With it, a cut is taken where the estimate sees a clear gain.  (Not another shape uncut, for which
  // nobody would ask for workspace: its estimate kept copies from being made, and the launch then ran without either.  A UNet block of
  // 2 x 4096 tokens, 320 wide, q6p 255 / 251 us.)
  const char* knob = getenv("DT_DENSE_SPLIT");  // "never" | "always" (as often as can be; for tests); read at every call
  if (ws_bytes == 0 || (knob && knob[0] == 'n')) return base;
  if (knob && knob[0] == 'a') {
    TilePlan p = pal_fits_big ? (m_max <= 128 ? tnarrow : t256) : tall_ok && !wide ? ttall : base;
    if (p.tile == kTile128x128) return base;
    p.whole = 0;
    p.split = std::min(kMaxSplit, nk / 2);
    return p.split > 1 && p.bytes() <= std::min(ws_bytes, kDenseMaxWorkspace) ? p : base;
  }
  TilePlan best = base;
  // A clear gain: 5 %, and 4 us for launches of up to 30, where the second launch and the workspace of a cut cost the host some of it.
  double least = 0.95 * start;
  const auto consider = [&](const TilePlan& shape) {
    double t;
    const TilePlan p = best_split(shape, w0.qbits, pal_mode(shape), nk, step, expanded, ws_bytes, &t);
    if (p.split > 1 && t < least && (t > 30.0 || t < start - 4.0)) {
      least = *cost = t;
      best = p;
    }
  };
  if (pal_fits_big) {
    consider(t256);
    consider(tnarrow);
  } else if (tall_ok && !wide) {
    consider(ttall);
  }
  return best;
}

// DT_DENSE_EXPAND = "never" | "always" (wherever it can be) overrides the choice between packed weights and copies; for tests and
// measurements, read at every call.  DT_DENSE_SPLIT has no say in it.
static bool expand_knob(char first) {
  const char* knob = getenv("DT_DENSE_EXPAND");
  return knob && knob[0] == first;
}

// The layout of one launch on plain fp16 weights, the palettized ones among them copied to scratch first.  Returns false where
// that cannot be, or is not wanted.
static bool plan_copies(const HostGroup* hs, int n, int w_begin, int w_end, bool wide, size_t ws, TilePlan* plan, double* cost) {
  if (expand_knob('n')) return false;
  size_t bytes = 0;
  int64_t weights = 0, m_max = 0;
  int copies = 0;
  for (int gi = 0; gi < n; gi++) {
    m_max = std::max(m_max, hs[gi].M);
    for (int j = w_begin; j < (n > 1 ? hs[gi].n_weights : w_end); j++) {
      const dt_qx_weight& w = hs[gi].W[j];
      if (w.qbits == 16) continue;
      if (w.nib < kDepalMinNib || w.count > 0x7fffffff) return false;  // (the tiled kernel's 32-bit byte offsets)
      bytes += ((size_t)w.count * 2 + 255) & ~(size_t)255;
      weights += w.count;
      copies++;
    }
  }
  if (weights == 0 || bytes > ws || bytes > kDenseMaxExpand || (bytes > kDenseFewRowsExpand && m_max <= kDenseFewRows && !expand_knob('a'))) return false;
  dt_qx_weight f16 = hs[0].W[w_begin];
  f16.qbits = 16;
  *plan = plan_format(hs, n, w_begin, w_end, wide, std::min(ws - bytes, kDenseMaxWorkspace), f16, true, cost);
  plan->expand_bytes = bytes;
  plan->expanded = copies;
  // A copy costs 3.4 us and 0.44 per million weights, 0.65 where it outgrows the memory-side cache (28 M weights 13 us, 94 M
  // 61), and the plain launch on it takes 0.93 of its estimate (medians of 700 launches of 65 .. 8192 rows; 0.87 over the larger set
  // that plan_cost names).
  const double m = 1e-6 * (double)weights;
  *cost = 0.93 * *cost + 3.4 + 0.44 * m + 0.21 * std::max(0.0, m - 64.0);
  return true;
}

// The layout of one launch with `ws` bytes of scratch, of which `expand` says whether fp16 copies of the weights may go
// into them.
// The tiled kernel on palettized weights looks every weight up once per tile of rows, at a cost that no schedule hides: 0.6
// against 0.2 us a K-tile on 128 x 128 tiles, however few the rows.  us, packed / copied: 4608 x 3072 -> 3 x 3072 q6p 284 /
// 227, 1376 x 3072 -> 12288 q8p 158 / 131, 512 x 3072 -> 3072 q8p 47 / 26; and the other way round 188 x 3840 -> 3 x 8192 q6p
// 84 / 112, 579 x 256 -> 5376 q6p 9.8 / 12.1.  The gain has to be 5 %, and 2 us, which are the host's for a second launch, and more where
// the estimate of so small a gain does not hold: 0.75 us for each of the weights, with several of which a short call waits for the host,
// and 0.25 for every million of them, which with few rows take longer to copy; 6 at most.  (840 calls of random sizes whose estimate lies between 3
// and 6 us: with 2 for all 0.936 of the time of 6 for all, but one in five slower by 2 % and more, up to 1.49 -- us, 91 x 448 -> 6 x 64 q8p 18.8 /
// 12.6, 127 x 1024 -> 3 x 3776 q5p 27.7 / 19.7 --; with this 0.928 and one in twenty.)  Behind a LoRA layer's down projection, whose launch is made
// anyway, 2 us do (0.963 of the time of 6, 890 layers: 464 x 704 -> 3008 q8p 34 / 27).
static TilePlan plan_tiles(const HostGroup* hs, int n, int w_begin, int w_end, bool wide, size_t ws, bool expand, double* cost, bool beside_down = false) {
  const dt_qx_weight& w0 = hs[0].W[w_begin];
  const TilePlan packed = plan_format(hs, n, w_begin, w_end, wide, std::min(ws, kDenseMaxWorkspace), w0, false, cost);
  // (The estimate knows palettes in LDS.  Looked up in memory a launch takes four times as long, median of 1000 of them; priced like
  // the others, 219 x 1024 -> 3 x 7808 in q8 blocks of 2048 with a head epilogue stayed packed, 169 us instead of 37.)
  if (choose_pal_mode(w0.qbits, w0.nib, hs[0].K, packed.BM, packed.BN, packed.tiles) == kPalGlobal) *cost *= 4.0;
  TilePlan plain;
  double copied;
  if (!expand || w0.qbits == 16 || !plan_copies(hs, n, w_begin, w_end, wide, ws, &plain, &copied)) return packed;
  const double least = beside_down ? 2.0 : std::min(6.0, 2.0 + 0.75 * plain.expanded + 0.125e-6 * (double)plain.expand_bytes);
  if (!expand_knob('a') && !(copied < 0.95 * *cost && copied < *cost - least)) return packed;
  *cost = copied;
  return plain;
}

// End of the run of weights from i on that share a launch: at most kMaxWeights, of one format, all within the tiled
// kernels' alignment.  *fused: one of them wants its head epilogue fused.  mixed: plain fp16 weights may be among palettized
// ones of one format, all of which can be copied to fp16.
static int weight_run(const HostGroup& h, int i, bool* fused, bool mixed = false) {
  const dt_qx_weight* first = &h.W[i];
  int end = i;
  for (; end < h.n_weights && end - i < kMaxWeights; end++) {
    const dt_qx_weight& w = h.W[end];
    if (!h.w_tiled(end)) break;
    if (mixed) {
      if (w.qbits != 16 && (w.nib < kDepalMinNib || (first->qbits != 16 && (w.qbits != first->qbits || w.nib != first->nib)))) break;
      if (first->qbits == 16) first = &w;
    } else if (w.qbits != first->qbits || (w.qbits != 16 && w.nib != first->nib)) {
      break;
    }
    *fused = *fused || (h.wants_epi(end) && h.fusable(end));
  }
  return end;
}

// The weights from i on that go out in the next launch of the tiled kernel, and how.
struct NextLaunch {
  int end;
  bool fused = false;
  TilePlan plan;
};
static NextLaunch next_launch(const HostGroup& h, int i, size_t ws, bool expand) {
  NextLaunch l;
  double cost;
  l.end = weight_run(h, i, &l.fused);
  l.plan = plan_tiles(&h, 1, i, l.end, l.fused, ws, expand, &cost);
  if (!expand) return l;
  // Palettized weights and plain ones on the same X -- a LoRA layer's base and down projections -- in one launch, on copies of
  // the palettized ones, where that is no slower than one launch after the other, each of which costs the host 5 us
  // (4608 x 3072 -> 3072 q6p and 64 plain features: 91 and 18 us, together 82).
  NextLaunch all;
  all.end = weight_run(h, i, &all.fused, true);
  double together;
  if (all.end <= l.end || !plan_copies(&h, 1, i, all.end, all.fused, ws, &all.plan, &together)) return l;
  for (int j = l.end; j < all.end;) {
    bool fused = false;
    const int end = std::min(weight_run(h, j, &fused), all.end);
    double apart;
    plan_tiles(&h, 1, j, end, fused, ws, true, &apart);
    cost += apart + 5.0;
    j = end;
  }
  return together < cost || expand_knob('a') ? all : l;
}

// Scratch memory of a call, or none.
struct Workspace {
  uint8_t* ptr = nullptr;
  size_t bytes = 0;
  bool expand = false;  // also for fp16 copies of the weights
};

// Zeroes the counters of a K-split launch (a fill kernel, so that the launch can be captured in a graph).
__global__ void dense_zero_counters_kernel(int32_t* counters, int n) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) counters[i] = 0;
}

// qx: the launch's n_w weights.  down: a LoRA layer's down projection to go out ahead of it, or null.
static dt_status launch_plan(hipStream_t s, DenseArgs& a, int n_w, const TilePlan& plan, const Workspace& ws,
                             const dt_qx_weight* const* qx, const LoraDownArgs* down = nullptr) {
  a.whole_tiles = (int32_t)plan.whole;
  a.split = plan.split;
  a.partials = nullptr;
  a.counters = nullptr;
  const int n_counters = plan.split > 1 ? (int)(plan.tiles - plan.whole) * kSplitNodes : 0;
  if (plan.split > 1) {
    a.counters = reinterpret_cast<int32_t*>(ws.ptr + plan.expand_bytes);
    a.partials = reinterpret_cast<float*>(ws.ptr + plan.expand_bytes + plan.counter_bytes());
  }
  int qbits = qx[0]->qbits, mode;
  if (plan.expand_bytes > 0) {
    static_assert(kDepalMax >= kMaxWeights, "every weight of a launch may need a copy");
    DepalettizeMany d = {};
    d.counters = a.counters;
    d.n_counters = n_counters;
    uint8_t* out = ws.ptr;
    int64_t tiles = 0;
    const int granules = down ? kLoraCopyGranules : 256;  // of a tile
    for (int i = 0; i < n_w; i++) {
      if (qx[i]->qbits == 16) continue;
      qbits = qx[i]->qbits;
      d.nib = qx[i]->nib;
      d.w[d.n++] = {a.w[i].data, reinterpret_cast<uint16_t*>(out), qx[i]->count / 32, (int32_t)tiles};
      a.w[i].data = out;
      tiles += (qx[i]->count / 32 + granules - 1) / granules;
      out += ((size_t)qx[i]->count * 2 + 255) & ~(size_t)255;
    }
    for (int i = n_w; i < kMaxWeights; i++) a.w[i] = a.w[0];
    if (const dt_status st = down ? lora_down_copies_launch(s, *down, qbits, d, (int)tiles) : depalettize_many_launch(s, qbits, d, (int)tiles);
        st != DT_OK)
      return st;
    qbits = 16;
    mode = kPlainF16;
    a.nib = 32;
    a.pal_step = 1;
  } else {
    mode = choose_pal_mode(qbits, a.nib, a.k, plan.BM, plan.BN, plan.tiles);
    if (down)
      if (const dt_status st = lora_down_launch(s, *down); st != DT_OK) return st;
    if (plan.split > 1) {
      hipLaunchKernelGGL(dense_zero_counters_kernel, dim3((unsigned)((n_counters + 255) / 256)), dim3(256), 0, s, a.counters, n_counters);
      if (const dt_status st = launch_status(); st != DT_OK) return st;
    }
  }
  return launch_dense(s, a, plan.tile, qbits, mode);
}

// One validated problem with M > 0: weights that share (qbits, nib) and meet the
// tiled kernel's alignment go out in runs of up to kMaxWeights per launch, of the
// kernel that streams the weights where X has few rows, else of the tiled one; the
// rest take the any-shape kernel.
static dt_status run_group(hipStream_t s, const HostGroup& h, const Workspace& ws) {
  const int64_t M = h.M, K = h.K;
  const bool x_ok = h.x_ok();
  int i = 0;
  while (i < h.n_weights) {
    const dt_qx_weight& w0 = h.W[i];
    const int64_t n_rows0 = w0.count / K;
    if (!(x_ok && h.w_tiled(i))) {
      if (n_rows0 > 0) {
        DenseAnyArgs g = {};
        g.x = h.X;
        g.ldx = h.ldx;
        g.m = M;
        g.n = n_rows0;
        g.k = K;
        g.w = static_cast<const uint8_t*>(w0.data);
        g.w_bytes = w0.qbits == 16 ? w0.count * 2 : dt_qx_bytes(w0.qbits, w0.nib, w0.count);
        g.qbits = w0.qbits;
        g.nib = w0.nib;
        g.bias = h.bias ? h.bias[i] : nullptr;
        g.y = h.Y[i];
        g.ldy = h.ldy[i];
        g.scale = post_scale(h, i);
        if (h.post) {
          const dt_dense_post& p = h.post[i];
          g.add = p.addend;
          g.ld_add = p.ld_addend;
          g.act = p.activation;
          g.gate = p.gate;
          g.res = p.residual;
          g.ld_res = p.ld_residual;
          g.gate32 = p.gate_f32;
          g.mul = p.multiplicand;
          g.ld_mul = p.ld_multiplicand;
        }
        dt_status st = dense_any_launch(s, g);
        if (st != DT_OK) return st;
        if (h.wants_epi(i)) {
          st = epilogue_pass(s, h, i);
          if (st != DT_OK) return st;
        }
      }
      i++;
      continue;
    }
    // few rows: the kernel that streams the weights
    bool any_fused = false;
    const int run_end = weight_run(h, i, &any_fused);
    int64_t run_features = 0;
    for (int j = i; j < run_end; j++) run_features += h.W[j].count / K;
    if (const int fb = dense_rows_features(M, K, w0.qbits, w0.nib, run_features); fb > 0) {
      DenseArgs a;
      DenseGroup& g = a.g[0];
      g.x = h.X;
      g.ldx = h.ldx;
      g.m = (int32_t)M;
      g.tiles_m = 1;
      g.tile_begin = 0;
      g.w_begin = 0;
      int64_t tiles = 0;
      const int first = i;
      for (; i < run_end; i++) tiles += add_weight(a, i - first, h, i, (int)tiles, fb, false);
      if (tiles > 0x7fffffff) return DT_NO_KERNEL;
      g.w_end = i - first;
      g.tiles_n = a.total_tiles = (int32_t)tiles;
      finish_args(a, 1, i - first, K, w0);
      dt_status st = dense_rows_launch(s, a, w0.qbits, fb);
      for (int j = first; j < i && st == DT_OK; j++)
        if (h.wants_epi(j)) st = epilogue_pass(s, h, j);
      if (st != DT_OK) return st;
      continue;
    }
    const NextLaunch next = next_launch(h, i, ws.bytes, ws.expand);
    const TilePlan& plan = next.plan;
    const int BM = plan.BM, BN = plan.BN;
    const bool big = BN == 256;
    DenseArgs a;
    DenseGroup& g = a.g[0];
    g.x = h.X;
    g.ldx = h.ldx;
    g.m = (int32_t)M;
    g.tiles_m = (int)((M + BM - 1) / BM);
    g.tile_begin = 0;
    g.w_begin = 0;
    int tiles_n = 0, cnt = 0;
    const int first = i;
    const dt_qx_weight* qx[kMaxWeights];
    for (; i < next.end; i++, cnt++) {
      qx[cnt] = &h.W[i];
      tiles_n += add_weight(a, cnt, h, i, tiles_n, BN, big && h.wants_epi(i) && h.fusable(i));
    }
    g.w_end = cnt;
    g.tiles_n = tiles_n;
    if ((int64_t)g.tiles_m * tiles_n > 0x7fffffff) return DT_NO_KERNEL;
    a.total_tiles = g.tiles_m * tiles_n;
    finish_args(a, 1, cnt, K, w0);
    dt_status st = launch_plan(s, a, cnt, plan, ws, qx);
    if (st != DT_OK) return st;
    for (int j = first; j < i; j++)
      if (h.wants_epi(j) && !(big && h.fusable(j))) {
        st = epilogue_pass(s, h, j);
        if (st != DT_OK) return st;
      }
  }
  return DT_OK;
}

// ---- a LoRA layer -------------------------------------------------------------------------------------------------
// The intermediate of the low-rank branch, ahead of everything else in scratch.
static size_t lora_t_bytes(int64_t M, const dt_lora_pair& p) { return ((size_t)M * p.rank * (p.f32 ? 4 : 2) + 255) & ~(size_t)255; }

// Whether the layer is one launch of a tiled kernel with the branch in its epilogue, behind its down projection.  (Few rows, and what is
// off the tiled kernels' alignment, run as Dense calls of their own; so do fp16 pairs of ranks that are no multiple of 16.)
// In fp16 the down projection of many ranks, or of long rows, reads more than a compute unit's L1 can deliver, where the tiled kernel
// shares it in LDS, and the Dense calls run it beside the base projection.  us, Dense calls / here:
//   rank 16 (32): 4608 x 3072 -> 3072 q6p 104 / 95 (105 / 100), 1376 x 3072 -> 3072 q8p 58 / 52 (58 / 54), 512 x 3072 -> 3072 q6p 42 / 38 (42 / 39), 2016 x
//   1280 -> 1280 q6p 30 / 24 (30 / 27), 300 x 1280 -> 1280 q8p 28 / 22 (28 / 24), 4096 x 320 -> 320 q6p 22 / 17 (22 / 19), and the other way round, rank 32, 2206
//   x 4928 -> 320 45 / 53, rank 16, 100 x 5120 -> 1280 51 / 53; rank 64 and 128, with kernels for them: 929 x 3456 -> 704 40 / 54, 1432 x 832 -> 640 24
//   / 25, 1571 x 704 -> 832 24 / 32.
//   fp32, rank 32 (128): 4608 x 3072 -> 3072 128 / 113 (203 / 184), 512 x 3072 -> 3072 50 / 43 (54 / 54), 300 x 1280 -> 1280 44 / 26 (44 / 38).  With many ranks the
//   epilogue is most of it, and where few compute units have a second tile they are alone with its fp32 products: rank 128, 1331 x 1088 -> 3072 q6p
//   (264 tiles of 128 x 128) 51 / 65, 2305 x 1536 -> 1856 fp16 (285) 69 / 79, 1617 x 320 -> 3712 q6p (377) 50 / 57; of 256 x 256 4371 x 640 -> 4672 rank 96 (342) 127 / 143; and
//   otherwise 1334 x 832 -> 2816 q6p (242 of 128 x 128) 44 / 42, 2182 x 384 -> 3008 (432) 53 / 49, 3844 x 960 -> 4096 (992) 121 / 111: 0.92 of the time up to 256
//   tiles, level above 384.
static bool lora_fusable(const HostGroup& h, const dt_lora_pair& p) {
  if (h.M <= 0 || !h.x_ok() || !h.w_tiled(0)) return false;
  if (dense_rows_features(h.M, h.K, h.W[0].qbits, h.W[0].nib, h.W[0].count / h.K) > 0) return false;
  if (p.f32) {
    const auto tiles = [&](int64_t t) { return ((h.M + t - 1) / t) * ((h.W[0].count / h.K + t - 1) / t); };
    if (p.rank > 64 && ((h.K < 2560 && tiles(128) > kDenseCUs && tiles(128) <= kDenseCUs * 3 / 2) || (h.K < 1024 && tiles(256) > kDenseCUs))) return false;
    return h.M <= 0x3fffffff && p.rank <= 4096;
  }
  if (h.K > 4096 && (h.M < 512 || p.rank > 16)) return false;
  return p.rank % 16 == 0 && p.rank <= 32 && p.ld_up % 4 == 0 && (reinterpret_cast<uintptr_t>(p.down) & 15) == 0 &&
         (reinterpret_cast<uintptr_t>(p.up) & 7) == 0;
}

static dt_status validate_lora(const HostGroup& h, const dt_lora_pair* p) {
  if (const dt_status st = validate_group(h); st != DT_OK) return st;
  if (!p || !p->down || !p->up || p->rank <= 0 || p->ld_up < p->rank || (p->f32 != 0 && p->f32 != 1)) return DT_INVALID;
  if (!(p->scale == p->scale) || p->scale - p->scale != 0.f) return DT_INVALID;
  const uintptr_t odd = p->f32 ? 3 : 1;
  if ((reinterpret_cast<uintptr_t>(p->down) & odd) || (reinterpret_cast<uintptr_t>(p->up) & odd)) return DT_INVALID;
  if (h.post && (h.post->addend || h.post->multiplicand || post_scale(h, 0) != 1.0f)) return DT_INVALID;
  return DT_OK;
}

static dt_status run_lora(hipStream_t s, const HostGroup& h, const dt_lora_pair& p, uint8_t* scratch, size_t bytes) {
  const size_t t_bytes = lora_t_bytes(h.M, p);
  const Workspace ws{scratch + t_bytes, bytes - t_bytes, true};
  double cost;
  const TilePlan plan = plan_tiles(&h, 1, 0, 1, false, ws.bytes, true, &cost, true);
  DenseArgs a;
  DenseGroup& g = a.g[0];
  g.x = h.X;
  g.ldx = h.ldx;
  g.m = (int32_t)h.M;
  g.tiles_m = (int)((h.M + plan.BM - 1) / plan.BM);
  g.tile_begin = 0;
  g.w_begin = 0;
  g.w_end = 1;
  g.tiles_n = add_weight(a, 0, h, 0, 0, plan.BN, false);
  if ((int64_t)g.tiles_m * g.tiles_n > 0x7fffffff) return DT_NO_KERNEL;
  a.total_tiles = g.tiles_m * g.tiles_n;
  finish_args(a, 1, 1, h.K, h.W[0]);
  a.lora = DenseLora{scratch, p.up, p.rank, p.ld_up, p.rank, p.f32};
  const LoraDownArgs down{h.X, h.ldx, h.M, h.K, p.down, p.rank, p.f32, p.scale, scratch};
  const dt_qx_weight* const qx[1] = {h.W};
  return launch_plan(s, a, 1, plan, ws, qx, &down);
}

// All problems in one launch, when every X and weight meets the tiled kernel's alignment, they share K and the weight
// format, and at least one of them is large enough for a tile of 256.  Returns false if they do not fit.
static bool groups_fuse(const HostGroup* hs, int n) {
  if (n < 2 || n > kMaxGroups) return false;
  const dt_qx_weight& w0 = hs[0].W[0];
  int total_w = 0;
  bool big = false;
  for (int gi = 0; gi < n; gi++) {
    const HostGroup& h = hs[gi];
    if (h.K != hs[0].K || !h.x_ok()) return false;
    for (int i = 0; i < h.n_weights; i++) {
      const dt_qx_weight& w = h.W[i];
      if (!h.w_tiled(i) || w.qbits != w0.qbits || (w.qbits != 16 && w.nib != w0.nib)) return false;
      big = big || (h.M >= 1024 && w.count / h.K >= 256);
    }
    total_w += h.n_weights;
  }
  if (!big || total_w > kMaxWeights) return false;
  if (choose_pal_mode(w0.qbits, w0.nib, hs[0].K, 256, 256) == kPalGlobal &&
      choose_pal_mode(w0.qbits, w0.nib, hs[0].K, 128, 128) != kPalGlobal)
    return false;  // problem by problem, on the small tile with its per-row palette table
  // the kernel variant with the elementwise tail has no fused head epilogue: such problems do not share a launch
  bool any_post = false, any_epi = false;
  for (int gi = 0; gi < n; gi++) {
    any_post = any_post || hs[gi].post != nullptr;
    for (int i = 0; i < hs[gi].n_weights; i++) any_epi = any_epi || hs[gi].wants_epi(i);
  }
  if (any_post && any_epi) return false;
  int64_t tiles = 0;
  for (int gi = 0; gi < n; gi++)
    for (int i = 0; i < hs[gi].n_weights; i++) tiles += ((hs[gi].M + 127) / 128) * ((hs[gi].W[i].count / hs[gi].K + 127) / 128);
  return tiles <= 0x7fffffff / 8;
}

static dt_status run_groups_fused(hipStream_t s, const HostGroup* hs, int n, const Workspace& ws) {
  const dt_qx_weight& w0 = hs[0].W[0];
  double cost;
  const TilePlan plan = plan_tiles(hs, n, 0, 0, true, ws.bytes, ws.expand, &cost);
  const dt_qx_weight* qx[kMaxWeights];
  const int BM = plan.BM, BN = plan.BN;
  DenseArgs a;
  int cnt = 0;
  int64_t tiles = 0;
  for (int gi = 0; gi < n; gi++) {
    const HostGroup& h = hs[gi];
    DenseGroup& g = a.g[gi];
    g.x = h.X;
    g.ldx = h.ldx;
    g.m = (int32_t)h.M;
    g.tiles_m = (int)((h.M + BM - 1) / BM);
    g.tile_begin = (int32_t)tiles;
    g.w_begin = cnt;
    int tiles_n = 0;
    for (int i = 0; i < h.n_weights; i++, cnt++) {
      qx[cnt] = &h.W[i];
      tiles_n += add_weight(a, cnt, h, i, tiles_n, BN, h.wants_epi(i) && h.fusable(i));
    }
    g.w_end = cnt;
    g.tiles_n = tiles_n;
    tiles += (int64_t)g.tiles_m * tiles_n;
  }
  a.total_tiles = (int32_t)tiles;
  finish_args(a, n, cnt, hs[0].K, w0);
  dt_status st = launch_plan(s, a, cnt, plan, ws, qx);
  for (int gi = 0; gi < n && st == DT_OK; gi++)
    for (int i = 0; i < hs[gi].n_weights && st == DT_OK; i++)
      if (hs[gi].wants_epi(i) && !hs[gi].fusable(i)) st = epilogue_pass(s, hs[gi], i);
  return st;
}

// The most that a launch may ask for.
static size_t scratch_limit(bool expand) { return kDenseMaxWorkspace + (expand ? kDenseMaxExpand : 0); }

// The workspace that run_group would use for h.
static size_t group_workspace(const HostGroup& h, bool expand) {
  size_t need = 0;
  if (!h.x_ok()) return 0;
  for (int i = 0; i < h.n_weights;) {
    if (!h.w_tiled(i)) {
      i++;
      continue;
    }
    bool wide = false;
    int end = weight_run(h, i, &wide);
    int64_t features = 0;
    for (int j = i; j < end; j++) features += h.W[j].count / h.K;
    if (dense_rows_features(h.M, h.K, h.W[i].qbits, h.W[i].nib, features) == 0) {
      const NextLaunch next = next_launch(h, i, scratch_limit(expand), expand);
      need = std::max(need, next.plan.bytes());
      end = next.end;
    }
    i = end;
  }
  return need;
}

// The problems of a grouped call that have rows, validated.
static dt_status gather_groups(int32_t n_groups, const dt_dense_group* groups, HostGroup (&hs)[64], int& n) {
  if (n_groups < 0 || (n_groups > 0 && !groups)) return DT_INVALID;
  if (n_groups > 64) return DT_INVALID;
  n = 0;
  for (int i = 0; i < n_groups; i++) {
    const dt_dense_group& d = groups[i];
    const HostGroup h{d.M, d.K, d.X, d.ldx, d.W, d.n_weights, d.bias, d.Y, d.ldy, d.epi, d.post};
    dt_status st = validate_group(h);
    if (st != DT_OK) return st;
    if (h.M > 0) hs[n++] = h;
  }
  return DT_OK;
}

static dt_status run_groups(dt_stream stream, int32_t n_groups, const dt_dense_group* groups, const Workspace& ws) {
  HostGroup hs[64];
  int n = 0;
  if (const dt_status st = gather_groups(n_groups, groups, hs, n); st != DT_OK) return st;
  if (n == 0) return DT_OK;
  if (const dt_status ready = device_ready(); ready != DT_OK) return ready;
  hipStream_t s = as_stream(stream);
  if (groups_fuse(hs, n)) return run_groups_fused(s, hs, n, ws);
  for (int i = 0; i < n; i++) {
    const dt_status st = run_group(s, hs[i], ws);
    if (st != DT_OK) return st;
  }
  return DT_OK;
}

}  // namespace dt

DT_EXPORT dt_status dt_dense_qx_f16(dt_stream stream, int64_t M, int64_t K, const uint16_t* X, int64_t ldx,
                                    const dt_qx_weight* W, int32_t n_weights, const uint16_t* const* bias,
                                    uint16_t* const* Y, const int64_t* ldy, uint32_t flags) {
  return dt_dense_qx_heads_f16(stream, M, K, X, ldx, W, n_weights, bias, Y, ldy, nullptr, flags);
}

DT_EXPORT dt_status dt_dense_qx_heads_f16(dt_stream stream, int64_t M, int64_t K, const uint16_t* X, int64_t ldx,
                                          const dt_qx_weight* W, int32_t n_weights, const uint16_t* const* bias,
                                          uint16_t* const* Y, const int64_t* ldy, const dt_head_epilogue* epi,
                                          uint32_t flags) {
  using namespace dt;
  (void)flags;
  const HostGroup h{M, K, X, ldx, W, n_weights, bias, Y, ldy, epi, nullptr};
  dt_status st = validate_group(h);
  if (st != DT_OK) return st;
  if (M == 0) return DT_OK;
  if (const dt_status ready = device_ready(); ready != DT_OK) return ready;
  return run_group(as_stream(stream), h, Workspace{});
}

DT_EXPORT dt_status dt_dense_qx_post_f16(dt_stream stream, int64_t M, int64_t K, const uint16_t* X, int64_t ldx,
                                         const dt_qx_weight* W, int32_t n_weights, const uint16_t* const* bias,
                                         uint16_t* const* Y, const int64_t* ldy, const dt_dense_post* post,
                                         uint32_t flags) {
  using namespace dt;
  (void)flags;
  const HostGroup h{M, K, X, ldx, W, n_weights, bias, Y, ldy, nullptr, post};
  dt_status st = validate_group(h);
  if (st != DT_OK) return st;
  if (M == 0) return DT_OK;
  if (const dt_status ready = device_ready(); ready != DT_OK) return ready;
  return run_group(as_stream(stream), h, Workspace{});
}

DT_EXPORT dt_status dt_dense_qx_grouped_f16(dt_stream stream, int32_t n_groups, const dt_dense_group* groups,
                                            uint32_t flags) {
  (void)flags;
  return dt::run_groups(stream, n_groups, groups, dt::Workspace{});
}

static size_t groups_workspace(int32_t n_groups, const dt_dense_group* groups, bool expand) {
  using namespace dt;
  HostGroup hs[64];
  int n = 0;
  if (gather_groups(n_groups, groups, hs, n) != DT_OK || n == 0) return 0;
  if (groups_fuse(hs, n)) {
    double cost;
    return plan_tiles(hs, n, 0, 0, true, scratch_limit(expand), expand, &cost).bytes();
  }
  size_t need = 0;
  for (int i = 0; i < n; i++) need = std::max(need, group_workspace(hs[i], expand));
  return need;
}

DT_EXPORT size_t dt_dense_workspace_bytes(int32_t n_groups, const dt_dense_group* groups) {
  return groups_workspace(n_groups, groups, false);
}

DT_EXPORT size_t dt_dense_scratch_bytes(int32_t n_groups, const dt_dense_group* groups) {
  return groups_workspace(n_groups, groups, true);
}

DT_EXPORT dt_status dt_dense_qx_grouped_ws_f16(dt_stream stream, int32_t n_groups, const dt_dense_group* groups,
                                               uint32_t flags, void* workspace, size_t workspace_bytes) {
  (void)flags;
  if (reinterpret_cast<uintptr_t>(workspace) & 255) return DT_INVALID;
  return dt::run_groups(stream, n_groups, groups,
                        dt::Workspace{static_cast<uint8_t*>(workspace), workspace ? workspace_bytes : 0, false});
}

DT_EXPORT dt_status dt_dense_qx_grouped_scratch_f16(dt_stream stream, int32_t n_groups, const dt_dense_group* groups,
                                                    uint32_t flags, void* scratch, size_t scratch_bytes) {
  (void)flags;
  if (reinterpret_cast<uintptr_t>(scratch) & 255) return DT_INVALID;
  return dt::run_groups(stream, n_groups, groups,
                        dt::Workspace{static_cast<uint8_t*>(scratch), scratch ? scratch_bytes : 0, true});
}

DT_EXPORT size_t dt_lora_dense_scratch_bytes(int64_t M, int64_t K, const uint16_t* X, int64_t ldx, const dt_qx_weight* W, uint16_t* Y,
                                             int64_t ldy, const dt_dense_post* post, const dt_lora_pair* pair) {
  using namespace dt;
  const HostGroup h{M, K, X, ldx, W, 1, nullptr, &Y, &ldy, nullptr, post};
  if (validate_lora(h, pair) != DT_OK || !lora_fusable(h, *pair)) return 0;
  double cost;
  return lora_t_bytes(M, *pair) + plan_tiles(&h, 1, 0, 1, false, scratch_limit(true), true, &cost, true).bytes();
}

DT_EXPORT dt_status dt_lora_dense_f16(dt_stream stream, int64_t M, int64_t K, const uint16_t* X, int64_t ldx, const dt_qx_weight* W,
                                      const uint16_t* bias, uint16_t* Y, int64_t ldy, const dt_dense_post* post, const dt_lora_pair* pair,
                                      uint32_t flags, void* scratch, size_t scratch_bytes) {
  using namespace dt;
  (void)flags;
  const HostGroup h{M, K, X, ldx, W, 1, &bias, &Y, &ldy, nullptr, post};
  if (const dt_status st = validate_lora(h, pair); st != DT_OK) return st;
  if (M == 0) return DT_OK;
  if (!lora_fusable(h, *pair)) return DT_NO_KERNEL;
  if (reinterpret_cast<uintptr_t>(scratch) & 255) return DT_INVALID;
  if (!scratch || scratch_bytes < lora_t_bytes(M, *pair)) return DT_OOM;
  if (const dt_status ready = device_ready(); ready != DT_OK) return ready;
  return run_lora(as_stream(stream), h, *pair, static_cast<uint8_t*>(scratch), scratch_bytes);
}
