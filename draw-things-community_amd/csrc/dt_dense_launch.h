// Launchers of the tiled Dense kernels, instantiated once per index width in dt_dense_q<Q>.hip.
#pragma once
#include "dt_dense_f16.h"
#include "dt_dense_kernel.h"

namespace dt {

// Tile shapes the host side chooses between.
// (tokens x features; 256 x 128 exists for the palettes that only fit beside a 128-feature tile -- per-row tables of
// 128 and 256 entries -- and is instantiated for those index widths only; 192 x 256 for plain fp16 weights, where its rounds of
// workgroups come out fuller)
enum DenseTile : int { kTile128x128 = 0, kTile128x256 = 1, kTile256x256 = 2, kTile256x128 = 3, kTile192x256 = 4 };

template <int Q, int BM, int BN, bool POST, bool LORA, bool SPLIT>
static dt_status launch_tiled(hipStream_t s, const DenseArgs& a, int mode) {
  const int64_t rest = SPLIT ? a.total_tiles - a.whole_tiles : 0;
  dim3 grid((unsigned)(a.total_tiles - rest + rest * a.split)), block(512);
  if constexpr (Q == 16) {  // plain fp16 weight
    // pair slots: as many as fit where a workgroup has a compute unit to itself (up to 256 tiles of 128 x 128 and K over 256: in
    // a kernel of their own; else two slots let two of them share one)
    if constexpr (BM == 128 && BN == 256) {
      hipLaunchKernelGGL((dense_qx_kernel<8, BM, BN, kPlainF16, POST, SPLIT, 3, LORA>), grid, block, 0, s, a);
    } else if constexpr (BM == 128 && BN == 128) {
      if (grid.x <= 256 && a.k > 256) hipLaunchKernelGGL((dense_f16_kernel<POST, LORA>), grid, block, 0, s, a);
      else hipLaunchKernelGGL((dense_qx_kernel<8, BM, BN, kPlainF16, POST, SPLIT, 2, LORA>), grid, block, 0, s, a);
    } else {
      hipLaunchKernelGGL((dense_qx_kernel<8, BM, BN, kPlainF16, POST, SPLIT, 2, LORA>), grid, block, 0, s, a);
    }
    return launch_status();
  } else {
    switch (mode) {
      case kPalShared:
        if constexpr (BM == 256 && BN == 128) return DT_NO_KERNEL;
        else hipLaunchKernelGGL((dense_qx_kernel<Q, BM, BN, kPalShared, POST, SPLIT, 2, LORA>), grid, block, 0, s, a);
        break;
      case kPalRow:
        if constexpr ((BN << (Q + 1)) <= pal_lds_bytes(BM, BN, kPalRow)) {
          hipLaunchKernelGGL((dense_qx_kernel<Q, BM, BN, kPalRow, POST, SPLIT, 2, LORA>), grid, block, 0, s, a);
          break;
        } else {
          return DT_NO_KERNEL;  // choose_pal_mode never picks per-row palettes that do not fit
        }
      default:
        if constexpr (BM == 256 && BN == 128) return DT_NO_KERNEL;
        else hipLaunchKernelGGL((dense_qx_kernel<Q, BM, BN, kPalGlobal, POST, SPLIT, 2, LORA>), grid, block, 0, s, a);
    }
    return launch_status();
  }
}

template <int Q, bool POST, bool LORA>
static dt_status launch_dense_qp(hipStream_t s, const DenseArgs& a, int tile, int mode) {
  switch (tile) {
    case kTile128x128: return launch_tiled<Q, 128, 128, POST, LORA, false>(s, a, mode);
    case kTile128x256:
      return a.partials ? launch_tiled<Q, 128, 256, POST, LORA, true>(s, a, mode) : launch_tiled<Q, 128, 256, POST, LORA, false>(s, a, mode);
    case kTile256x128:
      if constexpr (Q == 7 || Q == 8) {
        if (mode != kPalRow) return DT_NO_KERNEL;
        return a.partials ? launch_tiled<Q, 256, 128, POST, LORA, true>(s, a, mode) : launch_tiled<Q, 256, 128, POST, LORA, false>(s, a, mode);
      } else {
        return DT_NO_KERNEL;  // the host side picks this tile for 7- and 8-bit indices only
      }
    case kTile192x256:
      if constexpr (Q == 16) return a.partials ? DT_NO_KERNEL : launch_tiled<Q, 192, 256, POST, LORA, false>(s, a, mode);  // (never cut)
      else return DT_NO_KERNEL;
    default:
      return a.partials ? launch_tiled<Q, 256, 256, POST, LORA, true>(s, a, mode) : launch_tiled<Q, 256, 256, POST, LORA, false>(s, a, mode);
  }
}

// Every tiled kernel for Q-bit indices (Q = 16: plain fp16 weights); `post` selects the variant with the
// elementwise tail, which has one of its own with a LoRA layer's branch: skipped at run time it costs other tails 2 .. 5 % of a
// launch (us, GELU on plain weights, 256 x 256 tiles: 3346 x 1408 -> 2 x 4032 104 / 98.5, 8001 x 192 -> 3 x 1152 47.0 / 44.5).
// Instantiated once per Q in dt_dense_q<Q>.hip.
template <int Q>
dt_status launch_dense_q(hipStream_t s, const DenseArgs& a, int tile, bool post, int mode) {
  if (a.lora.up) return launch_dense_qp<Q, true, true>(s, a, tile, mode);
  return post ? launch_dense_qp<Q, true, false>(s, a, tile, mode) : launch_dense_qp<Q, false, false>(s, a, tile, mode);
}

}  // namespace dt
