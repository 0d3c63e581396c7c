// The dense 2 x 2-wave kernels of the wide (prefill) GEMM: gemm_tile.h's tile behind the wide
// kernel's grid (K splits into fragment-ordered tile blocks, the one-launch hybrid).
#include "gemm_tile.h"

namespace mxl {

// Stages of the LDS ring.  SHARED: of the workgroups that share a CU (RESIDENT of them); LONE:
// where the launch has too few for that, four, so that they keep as much in flight.
template <int MT, int NT>
struct TileDepth {
  static constexpr int RESIDENT = MT * NT > 16 ? 1 : MT * NT > 4 ? 2 : 4;
  static constexpr int SHARED = MT * NT > 32 || MT * NT == 16 || MT * NT == 4 ? 2 : 3;
  static constexpr int LONE = MT * NT > 16 ? SHARED : 4;
  // most workgroups per CU that still leave room for LONE stages each
  static constexpr int LONE_MAX = MT * NT == 4 ? 2 : 1;
  // of a tile's quarters, in the LDS of the launch
  static constexpr int QUARTER = 4;
};

template <int FMT, int MT, int NT, bool BLOCK>
struct WideKernel<FMT, MT, NT, BLOCK, false, 2> {
  static __device__ __forceinline__ void run(const GemmParams& p, const WideGrid& g) {
    constexpr int MTW = MT / 2, NTW = 2 * NT, BM = 16 * MT, TW = 64 * NT;
    extern __shared__ __attribute__((aligned(16))) uint8_t lds[];  // TileLds::bytes(g.depth)
    const int M = (int)p.M, KT = (int)p.KT;
    auto a_row = [&](int row) { return row < M ? row : M - 1; };
    const uint8_t* const sw = static_cast<const uint8_t*>(p.sw);
    // (32-bit indices: the host bounds the grid, and so every product below)
    const uint32_t L = blockIdx.x, tail0 = (uint32_t)g.tail0, rem_tiles = (uint32_t)g.rem_tiles;
    const uint32_t mblocks = (uint32_t)g.mblocks, nblocks = (uint32_t)g.nblocks, group_m = (uint32_t)g.group_m;
    // workgroups past the whole tiles: quarters of the last ones (whole K), or K splits of them
    const bool past = L >= tail0;
    uint32_t mb, nb;
    if constexpr (MT >= 8 && NT >= 2) {
      if (past && rem_tiles == 0) {
        const uint32_t unit = wide_logical(L - tail0, (uint32_t)gridDim.x - tail0);
        wide_coords(tail0 + (unit >> 2), mblocks, nblocks, group_m, mb, nb);
        const int row0 = (int)(mb * BM + (unit & 1) * (BM / 2)), qn = (int)(2 * nb + (unit >> 1 & 1));
        if (row0 >= M || (int64_t)qn * (TW / 2) >= p.N) return;
        const TileWork w{row0, M, qn, 0, KT, p.w, sw, nullptr};
        tile_gemm<FMT, MTW / 2, NTW / 2, BLOCK, TileDepth<MT, NT>::QUARTER>(p, w, lds, a_row);
        return;
      }
    }
    // tile of this workgroup, its K split of kps super-tiles, the split's partials
    const uint32_t at = past ? L - tail0 : wide_logical(L, tail0), tiles = past ? rem_tiles : (uint32_t)g.tiles;
    const uint32_t split = at / tiles, kps = (uint32_t)(past ? g.kt2 : g.kt_per_split);
    wide_coords((past ? tail0 : 0) + at - split * tiles, mblocks, nblocks, group_m, mb, nb);
    const int kb = (int)(split * kps), ke = kb + (int)kps < KT ? kb + (int)kps : KT;
    const TileWork w{(int)(mb * BM), M, (int)nb, kb, ke, p.w, sw,
                     past || p.S > 1 ? p.partial + (int64_t)at * (BM * TW) : nullptr};
    using D = TileDepth<MT, NT>;
    if (D::LONE != D::SHARED && g.depth == D::LONE) tile_gemm<FMT, MTW, NTW, BLOCK, D::LONE>(p, w, lds, a_row);
    else tile_gemm<FMT, MTW, NTW, BLOCK, D::SHARED>(p, w, lds, a_row);
  }
};

template <int FMT, bool BLOCK>
static hipError_t launch_tiles_fmt(const WideConfig& c, const GemmParams& p, const WideGrid& g0, int64_t grid,
                                   hipStream_t s) {
  const dim3 gr((unsigned)grid), blk(256);
  WideGrid g = g0;
#define MXL_TILES(MT_, NT_)                                                                              \
  if (c.MT == MT_ && c.NT == NT_) {                                                                      \
    using D = TileDepth<MT_, NT_>;                                                                       \
    using L = TileLds<MT_ / 2, 2 * NT_, BLOCK>;                                                          \
    static_assert(D::RESIDENT * L::bytes(D::SHARED) <= 160 * 1024, "the resident workgroups' LDS");      \
    static_assert(D::LONE_MAX * L::bytes(D::LONE) <= 160 * 1024, "the lone workgroups' LDS");            \
    using Q = TileLds<(MT_ > 4 ? MT_ / 4 : 2), (NT_ > 1 ? NT_ : 2), BLOCK>;                              \
    static_assert(MT_ < 8 || NT_ < 2 || Q::bytes(D::QUARTER) <= L::bytes(D::SHARED), "a quarter's LDS"); \
    g.depth = grid <= (int64_t)D::LONE_MAX * cu_count() ? D::LONE : D::SHARED;                           \
    hipLaunchKernelGGL((gemm_wide_kernel<FMT, MT_, NT_, BLOCK, false, 2>), gr, blk,                      \
                       (unsigned)L::bytes(g.depth), s, p, g);                                            \
    return hipGetLastError();                                                                            \
  }
  if constexpr (!BLOCK) {  // (the folds of block-FP8 keep its sums in the 256 addressable vector registers)
    MXL_TILES(16, 4)
    MXL_TILES(8, 4)
  }
  MXL_TILES(8, 2)
  MXL_TILES(8, 1)
  MXL_TILES(4, 2)
  MXL_TILES(4, 1)
#undef MXL_TILES
  return hipErrorInvalidValue;
}

hipError_t launch_wide_tiles(int fmt, bool block, const WideConfig& c, const GemmParams& p, const WideGrid& g,
                             int64_t grid, hipStream_t s) {
  if (grid > 0x7FFFFFFF) return hipErrorInvalidValue;
  if (block) return fmt == kE4M3 ? launch_tiles_fmt<kE4M3, true>(c, p, g, grid, s) : hipErrorInvalidValue;
  if (fmt == kE4M3) return launch_tiles_fmt<kE4M3, false>(c, p, g, grid, s);
  if (fmt == kE2M3) return launch_tiles_fmt<kE2M3, false>(c, p, g, grid, s);
  if (fmt == kE3M2) return launch_tiles_fmt<kE3M2, false>(c, p, g, grid, s);
  return hipErrorInvalidValue;
}

}  // namespace mxl
