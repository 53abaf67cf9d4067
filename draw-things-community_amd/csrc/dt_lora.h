// Launchers of a LoRA layer's down projections (dt_lora.hip).
#pragma once
#include "dt_common.h"
#include "dt_depalettize.h"

namespace dt {

// T[M, rank] = scale * (X[M, K] down[rank, K]^T), fp32 or rounded to fp16 before and behind the scale.
struct LoraDownArgs {
  const uint16_t* x;
  int64_t ldx, m, k;
  const void* down;
  int32_t rank;
  int32_t f32;
  float scale;
  void* t;  // row stride rank
};

dt_status lora_down_launch(hipStream_t s, const LoraDownArgs& a);
// The same, and palettized weights written out as fp16 (`tiles` tiles of kLoraCopyGranules granules) by the workgroups behind.
constexpr int kLoraCopyGranules = 512;
dt_status lora_down_copies_launch(hipStream_t s, const LoraDownArgs& a, int qbits, const DepalettizeMany& d, int tiles);

}  // namespace dt
