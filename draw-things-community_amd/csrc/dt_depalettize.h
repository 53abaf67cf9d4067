// Palettized weights written out as fp16 (dt_depalettize.hip): a workgroup's share, and the launcher of the kernel that does it
// ahead of a Dense.
#pragma once
#include "dt_common.h"
#include "dt_layout.h"

namespace dt {

constexpr int kDepalMinNib = 512;  // smallest block of the kernels that keep palettes in LDS
constexpr int kDepalMax = 8;       // weights per launch
// LDS of depalettize_tile: what its threads write, and their palettes.
constexpr int depalettize_lds(int Q, int NT) { return NT * 64 + ((32 * NT / kDepalMinNib + 2) << (Q + 1)); }

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

// The same granule-per-thread unpacking for blocks of 512 elements and more, with both sides of the lookup moved
// into LDS: the palettes of the (at most 32 NT / nib + 2) blocks that a workgroup's NT granules touch are loaded once,
// and the 64 bytes a thread produces go through a [thread][4 chunks] staging array, so that every store
// instruction of a wave writes 1 KB of consecutive addresses (thread-per-granule stores are 64 bytes apart per lane).
// Chunk c of thread t is staged at chunk 4 t + (c ^ (t / 4 % 4)): 16 consecutive lanes hit 16 different 16-byte
// bank groups on the way in (stride of 4 chunks) and on the way out (consecutive chunks).
// A thread's indices are asked for ahead of the palettes, so that the two memory latencies are one.
// tile: which NT granules of the tensor; NT: threads of the workgroup; smem: depalettize_lds(Q, NT) bytes of LDS, 16-byte aligned.
template <int Q, int NT>
__device__ __forceinline__ void depalettize_tile(const uint8_t* __restrict__ packed, int nib, int64_t n_granules,
                                                 int64_t tile, uint16_t* __restrict__ out, unsigned char* smem) {
  uint4_t* const stage = reinterpret_cast<uint4_t*>(smem);
  uint16_t* const pal = reinterpret_cast<uint16_t*>(smem + NT * 64);
  const int t = threadIdx.x;
  const int64_t g0 = tile * NT;
  const QxLayout l = make_layout(Q, nib);
  const int64_t g_last = (g0 + NT - 1 < n_granules ? g0 + NT - 1 : n_granules - 1);
  const int64_t b_first = g0 * 32 / nib, b_last = (g_last * 32 + 31) / nib;
  const int n_pal = (int)(b_last - b_first + 1);
  const int64_t g = g0 + t < n_granules ? g0 + t : g_last;
  const int64_t b = b_first + (uint32_t)(g * 32 - b_first * nib) / (uint32_t)nib;  // (the difference is below 32 NT + nib)
  const uint32_t* src = reinterpret_cast<const uint32_t*>(packed + index_byte_offset(l, b, g * 32 - b * nib));
  uint32_t raw[Q];
#pragma unroll
  for (int i = 0; i < Q; i++) raw[i] = src[i];
  for (int i = t; i < n_pal << (Q - 1); i += NT) {
    const int p = i >> (Q - 1), e = i & ((1 << (Q - 1)) - 1);
    reinterpret_cast<uint32_t*>(pal)[i] =
        reinterpret_cast<const uint32_t*>(packed + palette_offset(l, b_first + p))[e];
  }
  __syncthreads();
  {
    uint32_t idx[32];
    unpack32<Q>(raw, idx);
    const uint16_t* mine = pal + ((int)(b - b_first) << Q);
    uint32_t o[16];
#pragma unroll
    for (int j = 0; j < 16; j++) o[j] = (uint32_t)mine[idx[2 * j]] | ((uint32_t)mine[idx[2 * j + 1]] << 16);
#pragma unroll
    for (int c = 0; c < 4; c++)
      stage[4 * t + (c ^ ((t >> 2) & 3))] = uint4_t{o[4 * c], o[4 * c + 1], o[4 * c + 2], o[4 * c + 3]};
  }
  __syncthreads();
  // chunk L of the workgroup's 64 NT bytes (L = 4 * thread + c) leaves through lane L % NT of trip L / NT
  uint4_t* dst = reinterpret_cast<uint4_t*>(out + g0 * 32);
  const int64_t n_chunks = (g_last - g0 + 1) * 4;
#pragma unroll
  for (int j = 0; j < 4; j++) {
    const int L = j * NT + t;
    const int src_t = L >> 2, c = L & 3;
    if (L < n_chunks) dst[L] = stage[4 * src_t + (c ^ ((src_t >> 2) & 3))];
  }
}

dt_status depalettize_many_launch(hipStream_t s, int qbits, const DepalettizeMany& a, int tiles);

}  // namespace dt
