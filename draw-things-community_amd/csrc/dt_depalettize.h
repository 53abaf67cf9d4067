// Launcher of the kernel that writes palettized weights out as fp16 ahead of a Dense (dt_depalettize.hip).
#pragma once
#include "dt_common.h"

namespace dt {

constexpr int kDepalMinNib = 512;  // smallest block of the kernels that keep palettes in LDS
constexpr int kDepalMax = 8;       // weights per launch

// Weights of one format (nib a multiple of 32, at least kDepalMinNib; counts multiples of 32), their tiles of 256
// granules numbered one weight after the other; packed 4-byte and out 16-byte aligned.
struct DepalettizeMany {
  int32_t nib, n;
  int32_t* counters;  // [n_counters] zeroed
  int32_t n_counters;
  struct {
    const uint8_t* packed;
    uint16_t* out;
    int64_t n_granules;
    int32_t tile_begin;
  } w[kDepalMax];
};

dt_status depalettize_many_launch(hipStream_t s, int qbits, const DepalettizeMany& a, int tiles);

}  // namespace dt
