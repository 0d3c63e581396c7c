// The grouped (MoE) kernel of the wide GEMM: gemm_tile.h's 2 x 2-wave tiles over the routed
// rows of every expert.
//
// Persistent workgroups, two per CU, walk the (m-block, n-block) tiles of the routed rows: every
// workgroup scans the experts' 16 MT-row block counts once, thread t keeping experts 4 t .. 4 t + 3,
// and the thread that holds a tile's block hands over its expert, so the launch needs no host-side
// counts and experts without rows read no weights.  n-blocks are walked fastest (an expert block's
// gathered rows stay in one XCD's L2 over its n-blocks).  A block of at most 64 rows (an expert's
// last block) runs 64-row tiles: half the activation copies and MFMAs.
//
// The experts' weights bound it: W6A8 256 experts of 1024 x 2048, 64 rows each on average, 403 MB
// of weights, 118 us with the four-wave tiles, 106.1 with these (3.8 TB/s; 106.5 with each tile's
// rows looked up at its start instead of under the K walk of the tile before it).
#include "gemm_tile.h"

namespace mxl {

// Stages of the LDS ring of a block's tile, as many as two workgroups per CU have room for.
template <int MT>
struct GroupedDepth {
  static constexpr int value = MT == 8 ? 2 : 3;
};

template <int FMT, int MT, int NT>
struct WideKernel<FMT, MT, NT, false, true, 1> {
  static __device__ __forceinline__ void run(const GemmParams& p, const WideGrid& g) {
    constexpr int BM = 16 * MT, EPT = (int)kWideGroupedMaxExperts / 256;  // experts per thread
    extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
    __shared__ int4 sh_tile[2];         // of this tile and the next: expert, first row, end of its rows
    __shared__ int32_t sh_row[2][BM];   // their activation rows
    __shared__ int32_t sh_wave[4];
    const int t = threadIdx.x, lane = t & 63, wv = t >> 6;
    const int E = (int)g.num_experts;

    // first m-blocks of this thread's experts e0 .. e0 + EPT - 1: their block counts scanned
    // over the wavefront and the four of them
    const int e0 = t * EPT;
    int pre[EPT + 1], row[EPT + 1];
    pre[0] = 0;
#pragma unroll
    for (int j = 0; j <= EPT; ++j) row[j] = (int)p.expert_offsets[e0 + j < E ? e0 + j : E];  // none past E
#pragma unroll
    for (int j = 0; j < EPT; ++j) pre[j + 1] = pre[j] + (row[j + 1] - row[j] + BM - 1) / BM;
    int sum = pre[EPT];
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
      const int v = __shfl_up(sum, d, 64);
      if (lane >= d) sum += v;
    }
    if (lane == 63) sh_wave[wv] = sum;
    __syncthreads();
    int base = sum - pre[EPT], total = 0;
    for (int v = 0; v < 4; ++v) {
      if (v < wv) base += sh_wave[v];
      total += sh_wave[v];
    }
    total = __builtin_amdgcn_readfirstlane(total);
    const uint32_t nblocks = (uint32_t)g.nblocks, blocks = total < g.mblocks ? (uint32_t)total : (uint32_t)g.mblocks;
    const uint32_t tiles = blocks * nblocks;
    if (blockIdx.x >= tiles) return;
    // Tile L: the thread that holds its expert hands over the expert and its row range
    auto find = [&](uint32_t L, int slot) {
      const int at = (int)(wide_logical(L, tiles) / nblocks) - base;
#pragma unroll
      for (int j = 0; j < EPT; ++j)
        if (pre[j] <= at && at < pre[j + 1])
          sh_tile[slot] = make_int4(e0 + j, row[j] + (at - pre[j]) * BM, row[j + 1], 0);
    };
    // activation row of thread t's row of the tile (past the expert's last: that one)
    auto gather = [&](const int4& x) -> int {
      const int r = x.y + t < x.z ? x.y + t : x.z - 1;
      return t >= BM ? 0 : p.row_index ? p.row_index[r] / p.row_div : r;
    };
    auto tile_of = [&](int slot) -> int4 {
      const int4 x = sh_tile[slot];
      return make_int4(__builtin_amdgcn_readfirstlane(x.x), __builtin_amdgcn_readfirstlane(x.y),
                       __builtin_amdgcn_readfirstlane(x.z), 0);
    };
    find(blockIdx.x, 0);
    __syncthreads();
    int4 x = tile_of(0);
    if (t < BM) sh_row[0][t] = gather(x);
    int buf = 0;
    for (uint32_t L = blockIdx.x; L < tiles; L += gridDim.x) {
      // the next tile's rows are looked up under this one's K walk
      const uint32_t next = L + gridDim.x;
      if (next < tiles) find(next, buf ^ 1);
      __syncthreads();  // (also ends the previous tile's reads of the ring)
      int4 y = x;
      int ahead = 0;
      if (next < tiles) {
        y = tile_of(buf ^ 1);
        ahead = gather(y);
      }
      const uint32_t logical = wide_logical(L, tiles);
      const TileWork w{x.y, x.z, (int)(logical % nblocks), 0, (int)p.KT, p.w + x.x * p.w_expert_stride,
                       static_cast<const uint8_t*>(p.sw) + x.x * p.sw_expert_stride, nullptr};
      const int* const rows = sh_row[buf];
      auto a_row = [&](int r) -> int { return rows[r - x.y]; };
      if (MT == 8 && x.z - x.y <= 64) tile_gemm<FMT, 2, 2 * NT, false, GroupedDepth<4>::value>(p, w, lds, a_row);
      else tile_gemm<FMT, MT / 2, 2 * NT, false, GroupedDepth<MT>::value>(p, w, lds, a_row);
      buf ^= 1;
      if (t < BM) sh_row[buf][t] = ahead;
      x = y;
    }
  }
};

template <int FMT, int MT, int NT>
static hipError_t launch_grouped_tile(const GemmParams& p, const WideGrid& g, int64_t grid, hipStream_t s) {
  constexpr int whole = TileLds<MT / 2, 2 * NT, false>::bytes(GroupedDepth<MT>::value);
  constexpr int half = TileLds<2, 2 * NT, false>::bytes(GroupedDepth<4>::value);
  constexpr int bytes = whole > half ? whole : half;
  static_assert(2 * (bytes + 1088) <= 160 * 1024, "two workgroups per CU");
  hipLaunchKernelGGL((gemm_wide_kernel<FMT, MT, NT, false, true, 1>), dim3((unsigned)grid), dim3(256), bytes, s, p, g);
  return hipGetLastError();
}

template <int FMT>
static hipError_t launch_grouped_fmt(const WideConfig& c, const GemmParams& p, const WideGrid& g, int64_t grid,
                                     hipStream_t s) {
  if (c.NT != 2) return hipErrorInvalidValue;
  if (c.MT == 8) return launch_grouped_tile<FMT, 8, 2>(p, g, grid, s);
  if (c.MT == 4) return launch_grouped_tile<FMT, 4, 2>(p, g, grid, s);
  return hipErrorInvalidValue;
}

hipError_t launch_wide_grouped(int fmt, const WideConfig& c, const GemmParams& p, const WideGrid& g, int64_t grid,
                               hipStream_t s) {
  if (fmt == kE4M3) return launch_grouped_fmt<kE4M3>(c, p, g, grid, s);
  if (fmt == kE2M3) return launch_grouped_fmt<kE2M3>(c, p, g, grid, s);
  if (fmt == kE3M2) return launch_grouped_fmt<kE3M2>(c, p, g, grid, s);
  return hipErrorInvalidValue;
}

}  // namespace mxl
