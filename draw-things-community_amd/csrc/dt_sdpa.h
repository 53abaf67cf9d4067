// Internal argument block of the attention kernel.
#pragma once
#include "dt_common.h"

namespace dt {

constexpr int kMaxSeg = 4;

struct SdpaSeg {
  const uint16_t* ptr;
  int64_t sb, ss, sh;
  int64_t start;  // first joint position of this segment
};

struct SdpaArgs {
  int32_t B, Hq, Hk, group, D;
  int64_t Sq, Skv;
  int32_t n_qseg, n_kvseg;
  SdpaSeg q[kMaxSeg], k[kMaxSeg], v[kMaxSeg];
  uint16_t* o;
  int64_t o_sb, o_ss, o_sh;
  float scale_log2e;
  // Optional per-head RMSNorm and RoPE rotation of the queries, applied to the query fragments on their way into
  // registers (same arithmetic and rounding as the norm / rotate pass): q_gamma[i] is segment i's norm weight [D]
  // or null, q_rot the table [joint query rows, D] or null.
  const uint16_t* q_gamma[kMaxSeg];
  const uint16_t* q_rot;
  float q_eps;
  int32_t q_prep;  // any of the above is set
  int32_t q_norm;     // any q_gamma is (filled by the launcher)
  int32_t q_aligned;  // q_rot and every q_gamma lie on 16 bytes (the same)
  // Key-split launch (optional; partials == nullptr runs one workgroup per task): workspace for the parts' partial
  // results and the counters of their meetings, sized and laid out by sdpa_split_plan().
  float* partials;
  int32_t* counters;
  int32_t whole_tasks;  // tasks with a workgroup each
  int32_t cut_tasks;    // the ones behind them, each cut along its keys into
  int32_t shares;       // this many parts
  int32_t counters_zeroed;  // by an earlier launch
  int32_t q_tiles, total_blocks;  // filled by the launcher
};

// Floats of one partial-result slot of the key-split kernel: 512 threads x DP / 32 * 16 accumulators, then for each wave the 32
// reference maxima and 32 row sums of its queries; the last 512 are spare, so that callers are asked for the room that they
// always were.
constexpr int sdpa_split_slot_floats(int dp) { return (dp / 32) * 16 * 512 + 2 * 512; }

// Most parts of a task; their meetings are 4 + 2 + 1.
constexpr int kSdpaSplitNodes = 8;

// How a launch would be split along the keys, and the workspace that takes.
struct SdpaSplit {
  int32_t whole_tasks;    // of the B * Hq * ceil(Sq / 256) tasks, full rounds of which stay whole
  int32_t cut_tasks;      // the others, each cut into
  int32_t shares;         // this many parts
  size_t counter_bytes;   // counters of the cut tasks (256-byte aligned), followed by
  size_t partial_bytes;   // a slot per part
  size_t room;            // workspace to ask callers for (at least bytes())
  size_t bytes() const { return counter_bytes + partial_bytes; }
};
// True when splitting pays: the task count leaves a good part of the last round of workgroups idle and there are enough
// key tiles to cut.  Uses the compute-unit count of the calling thread's current device.
bool sdpa_split_plan(int32_t B, int32_t Hq, int32_t D, int64_t Sq, int64_t Skv, SdpaSplit* plan);

dt_status sdpa_launch(hipStream_t s, const SdpaArgs& a);

// Device address of the current device's static scratch array (the one dt_sdpa_f16_static uses); looked up once
// per device.  nullptr on failure.
void* sdpa_static_scratch();

}  // namespace dt
