// Argument block and launcher of the any-shape Dense kernel (dt_dense_any.hip).
#pragma once
#include "dt_common.h"
#include "dt_dense_any_index.h"

namespace dt {

// One weight of one problem, with its tail.  Nothing is assumed about widths, block size or alignment.
struct DenseAnyArgs {
  const uint16_t* x;
  int64_t ldx;
  int64_t m, n, k;
  const uint8_t* w;
  int64_t w_bytes;  // bytes of the packed buffer (plain fp16: of the tensor)
  int32_t qbits, nib;
  const uint16_t* bias;
  uint16_t* y;
  int64_t ldy;
  float scale;
  const uint16_t* add;
  int64_t ld_add;
  int32_t act;
  const uint16_t* gate;
  float* res;
  int64_t ld_res;
  const float* gate32;
  const uint16_t* mul;
  int64_t ld_mul;
  // filled by the launcher
  int64_t tiles_m;
  int32_t pal_shared;  // the palettes of a tile's rows fit into LDS
};

dt_status dense_any_launch(hipStream_t s, DenseAnyArgs a);

}  // namespace dt
