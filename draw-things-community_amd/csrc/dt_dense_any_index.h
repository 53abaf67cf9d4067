// Where the any-shape Dense kernel (dt_dense_any.hip) reads a packed weight: which palettes the LDS of a tile holds, which
// block and which words a thread's run of 16 weights lies in.  Plain arithmetic, so that the host can check its bounds.
#pragma once
#include "dt_layout.h"

namespace dt {

constexpr int kAnyPalBytes = 16384;  // LDS for the palettes of a tile's rows (with a group's tiles: three workgroups per CU; with four groups' 64 x 64 tiles all of it)

// Rows past the last one read the last one: the only row that is sure to lie among the palettes of their tile.
DT_HD int64_t any_row(int64_t row, int64_t n) { return row < n ? row : n - 1; }

// The blocks that rows [n0, n0 + bt) of an [n, k] weight touch.
struct AnyBlocks {
  int64_t first;
  int count;
};
DT_HD AnyBlocks any_blocks(int64_t n0, int bt, int64_t n, int64_t k, int nib) {
  const int64_t first = n0 * k / nib;
  return AnyBlocks{first, (int)(((any_row(n0 + bt - 1, n) + 1) * k - 1) / nib - first + 1)};
}

// The palettes of any `bt` consecutive rows fit into the LDS set aside for them.
DT_HD bool any_pal_shared(int bt, int64_t k, int qbits, int nib) {
  return (bt * k / nib + 2) * ((int64_t)2 << qbits) <= kAnyPalBytes;
}

// Block and position in it of a thread's next run.
struct AnyCursor {
  int64_t blk;
  uint32_t r;
};
DT_HD AnyCursor any_cursor(int64_t row, int64_t k, int at, int nib) {
  const int64_t e = row * k + at, blk = e / nib;
  return AnyCursor{blk, (uint32_t)(e - blk * nib)};
}
DT_HD void any_advance(AnyCursor& c, uint32_t step, int nib) {
  c.r += step;
  if (c.r >= (uint32_t)nib) {
    const uint32_t q = c.r / (uint32_t)nib;
    c.blk += q;
    c.r -= q * (uint32_t)nib;
  }
}

// Weights of a 16-long run at k0 that exist, and those of them in the block where the run starts.
DT_HD int any_run(int64_t k0, int64_t k) { return k0 >= k ? 0 : (k - k0 < 16 ? (int)(k - k0) : 16); }
DT_HD int any_run_head(const AnyCursor& c, int run, int nib) {
  return (uint32_t)nib - c.r < (uint32_t)run ? (int)((uint32_t)nib - c.r) : run;
}

// Whole runs are fetched as words, unless blocks are shorter than a run (one may then touch more than two) or the buffer
// is shorter than a run's words.
DT_HD bool any_by_words(int words, int64_t w_bytes, int nib) { return nib >= 16 && w_bytes >= 4 * words; }

// First byte of the `words` dwords to fetch for byte p: the last runs of the buffer are read from further ahead instead of
// past its end.
DT_HD int64_t any_words_at(int64_t p, int words, int64_t w_bytes) { return p + 4 * words <= w_bytes ? p : w_bytes - 4 * words; }

// Bit at which the string starts in which the rest of a run -- beyond its first `head` weights, in the block after
// c.blk -- has the same place as in the run (the bits in between, palette bytes, are not looked at).
DT_HD int64_t any_rest_bit(const QxLayout& l, const AnyCursor& c, int head) {
  return (palette_offset(l, c.blk + 1) + l.pal_bytes) * 8 - (int64_t)head * l.qbits;
}

}  // namespace dt
