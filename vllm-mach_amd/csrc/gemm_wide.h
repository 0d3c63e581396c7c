// Declarations shared by the wide (prefill) GEMM's kernels: the four-wave tiles of
// gemm_wide.hip and the 2 x 2-wave tiles of gemm_tile.hip.
#pragma once

#include "gemm_common.h"

namespace mxl {

struct WideGrid {
  int64_t mblocks;       // dense: ceil(M / 16 MT); grouped: bound on sum_e ceil(rows_e / 16 MT)
  int64_t nblocks;       // ceil(N / (64 NT))
  int64_t kt_per_split;  // 512-wide super-tiles per split
  int64_t num_experts;   // grouped only
  int64_t tiles;         // dense: the output tiles this launch covers whole (numbered by wide_coords)
  // dense, one-launch hybrid: after its whole-K tile (tiles [0, tiles), bf16 out) workgroup
  // L also runs unit L < rem_tiles * S2 of the remainder: tile rem_tile0 + L % rem_tiles,
  // K split L / rem_tiles of kt2 super-tiles, into compact partials
  int64_t rem_tile0, rem_tiles, kt2;
  int S2;
  int64_t group_m;       // dense: m-blocks walked together
  // 2 x 2-wave tiles: workgroups from `tail0` on run what is left after `tail0` whole tiles (or
  // K splits of tiles): the quarters of the further tiles (four each, whole K), or with rem_tiles
  // the K splits of a hybrid's remainder.  Stages in the LDS ring.
  int64_t tail0;
  int depth;
};

// Block of tile `tile`: group_m m-blocks by all n-blocks at a time, m fastest.
template <class I>
__device__ __forceinline__ void wide_coords(I tile, I mblocks, I nblocks, I group_m, I& mb, I& nb) {
  const I gsz = group_m * nblocks, grp = tile / gsz, in = tile - grp * gsz;
  const I left = mblocks - grp * group_m, gm = left < group_m ? left : group_m;
  mb = grp * group_m + in % gm;
  nb = in / gm;
}

// Logical index of workgroup L of G: consecutive logical indices share an XCD (workgroup L
// runs on XCD L % 8) and so its L2.
template <class I>
__device__ __forceinline__ I wide_logical(I L, I G) {
  const I xcd = L & 7, per = G >> 3, extra = G & 7;
  return xcd * per + (xcd < extra ? xcd : extra) + (L >> 3);
}

// Workgroups per CU the kernel is compiled for: the 2 x 2-wave tiles by their size (LDS and
// registers), the grouped tiles two, the dense four-wave tiles one.
template <int MT, int NT, bool GROUPED, int WM>
struct WidePerCu {
  static constexpr int value = WM == 2 ? (MT * NT > 16 ? 1 : MT * NT > 8 ? 2 : 3) : GROUPED ? 2 : 1;
};

// Arrangement of the four waves: WM = 1 side by side (each all MT m-tiles by NT n-tiles;
// gemm_wide.hip), WM = 2 two by two (each MT / 2 m-tiles by 2 NT n-tiles; gemm_tile.hip).  Grouped
// launches (WM = 1 by name) are two by two as well (gemm_tile_grouped.hip).
template <int FMT, int MT, int NT, bool BLOCK, bool GROUPED, int WM>
struct WideKernel;

template <int FMT, int MT, int NT, bool BLOCK, bool GROUPED, int WM>
__global__ __launch_bounds__(256, (WidePerCu<MT, NT, GROUPED, WM>::value)) void gemm_wide_kernel(GemmParams p,
                                                                                               WideGrid g) {
  WideKernel<FMT, MT, NT, BLOCK, GROUPED, WM>::run(p, g);
}

// The dense 2 x 2-wave launch of `grid` workgroups.
hipError_t launch_wide_tiles(int fmt, bool block, const WideConfig& c, const GemmParams& p, const WideGrid& g,
                             int64_t grid, hipStream_t s);

// The grouped (MoE) launch of `grid` persistent workgroups (gemm_tile_grouped.hip).
hipError_t launch_wide_grouped(int fmt, const WideConfig& c, const GemmParams& p, const WideGrid& g, int64_t grid,
                               hipStream_t s);

}  // namespace mxl
