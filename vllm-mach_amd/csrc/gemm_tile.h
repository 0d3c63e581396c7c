// One output tile of the 2 x 2-wave GEMM on gfx950 (MX and block-FP8 weights): the device
// body of the dense kernels of gemm_tile.hip and the grouped ones of gemm_tile_grouped.hip.
//
// What bounds it.  At 128 x 128 tiles per workgroup every K128 stage moves as many LDS
// bytes as the LDS serves in the time of its MFMAs, so the wide kernel (gemm_wide.hip)
// stays near a fifth of the MFMA peak however its copies are scheduled.  Here four waves
// in a 2 x 2 arrangement own 16 MTW x 16 NTW outputs each (128 x 128 at MTW = NTW = 8, a
// 256 x 256 workgroup tile): per stage the LDS moves 128 KiB of fragment reads and 64 KiB
// of copies (1536 cycles at 128 bytes per cycle) under 2048 cycles of MFMAs, and each
// byte from L2 feeds twice the flops.
//
// Pipeline.  The operands of a stage arrive as four units, the upper and lower half of
// every wave's rows (A0, A1) and columns (B0, B1), each in its own LDS slot, two to four
// stages deep: as many as the workgroups of a CU leave room for, since the copies in flight are
// what a launch with cold weights waits on.  A stage is four quadrants of (MTW / 2) (NTW / 2) MFMAs, walked so
// that consecutive quadrants share one half:
//   even stages (A0,B0) (A0,B1) (A1,B1) (A1,B0), odd stages (A0,B1) (A0,B0) (A1,B0) (A1,B1)
// so one register copy of each half suffices: the unit a quadrant needs next is read from
// LDS while the previous quadrant's MFMAs run, into registers whose last use is behind it.
// Twice per stage a barrier hands over two units and frees the two slots read before it,
// into which the copies of `depth` stages ahead are issued (vmcnt counts them: loads complete
// in issue order), so all but half a stage of the ring is in flight.
//
// Measured, weights rotated out of the caches (us, the tiles of waves side by side or, where
// they do not run, the generic kernel before): W6A8 4096 x 17408 x 5120 665 -> 302 (2.4 PFLOP/s),
// 1024 x 17408 x 5120 150 -> 95, 48 x 17408 x 5120 51 -> 23.4 (2.9 TB/s of weights); block-FP8 512
// x 18432 x 2560 55.5 -> 36.2, 32 x 18432 x 2560 29.3 -> 13.5 (3.5 TB/s); MXFP8 512 x 2560 x 9216
// 27.9 -> 25.8.  The 256 x 256 tile is bound by its MFMAs at the clock that the power limit leaves (W6A8
// 4096 x 17408 x 5120: MFMAs busy 58 % of the cycles, 0.6 LDS reads each), the smaller ones by their LDS
// traffic (1.3 to 1.7 reads per MFMA; 8-byte FP6 reads with bank conflicts) and, in the last round, the
// epilogue.
//
// The weights take the MFMA's A operand and the activations its B operand, so a lane holds
// four consecutive output columns of one row (8-byte stores), and in block-FP8 its four
// sums share one activation scale.
#pragma once

#include "gemm_wide.h"

// the copies set M0 (the LDS base of a global->LDS load) themselves
#pragma clang diagnostic ignored "-Winline-asm"

namespace mxl {

typedef __attribute__((address_space(3))) uint8_t tile_lds_u8;

__device__ __forceinline__ uint32_t tile_lds(const uint8_t* p) { return (uint32_t)(uintptr_t)(const tile_lds_u8*)p; }

// Lane i copies 16 (4) bytes from base + voff to LDS [lds + 16 i] ([lds + 4 i]); base and
// lds are wave-uniform.
__device__ __forceinline__ void tile_copy16(const uint8_t* base, uint32_t voff, uint32_t lds) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(lds), "v"(voff), "s"(base) : "m0");
}
__device__ __forceinline__ void tile_copy4(const uint8_t* base, uint32_t voff, uint32_t lds) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dword %1, %2" ::"s"(lds), "v"(voff), "s"(base) : "m0");
}

// All but the newest N copies of this wave have landed and its LDS reads are done, then the
// barrier (no memory fence: it would drain the copies in flight).
template <int N>
__device__ __forceinline__ void tile_wait() {
  static_assert(N >= 0 && N <= 63, "vmcnt immediate");
  asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(N) : "memory");
}
// Piece permutation of row r (0..15) of an m-tile stored as whole 128-byte rows: piece p
// sits at 128 (r % 8) + 16 (p ^ tile_swz(r)) of its 1 KiB chunk, so that the fragment reads
// (lane 16 q + r: row r, pieces q and 4 + q) are free of bank conflicts.
__device__ __forceinline__ int tile_swz(int r) { return ((r >> 1) ^ ((r & 1) << 2)) & 7; }

template <int J>
struct Slice { static constexpr int value = J; };

typedef int v6i __attribute__((ext_vector_type(6)));
template <int FMT>
struct TileB { typedef v8i type; };
template <>
struct TileB<kE2M3> { typedef v6i type; };
template <>
struct TileB<kE3M2> { typedef v6i type; };

// c += W A^T for one 16 x 16 tile over a K128 slice, J the slice's byte of the packed E8M0
// operands.  Written as assembly so that the accumulator is updated in place: with 256
// accumulator registers live the compiler's allocator finds no room to rename one, and moves
// whole tiles between register files instead (measured on its output: several hundred moves
// and spills per stage).  The caller keeps two instructions between a VALU write of an
// operand and its use, and waits out the last MFMA before it or the compiler reads an accumulator
// (tests/test_mfma_hazards_host.py scans the built code for both).
template <int FMT, int J>
__device__ __forceinline__ void tile_mfma(v4f& c, const typename TileB<FMT>::type& w, const v8i& a, uint32_t sw,
                                          uint32_t sa) {
#define MXL_TILE_MFMA(SEL_, FMT_)                                                                                   \
  asm volatile("v_mfma_scale_f32_16x16x128_f8f6f4 %0, %1, %2, %0, %3, %4 " SEL_ FMT_                                \
               : "+a"(c) : "v"(w), "v"(a), "v"(sw), "v"(sa))
#define MXL_TILE_MFMA_J(FMT_)                                                              \
  if constexpr (J == 0) MXL_TILE_MFMA("op_sel_hi:[0,0,0]", FMT_);                          \
  else if constexpr (J == 1) MXL_TILE_MFMA("op_sel:[1,1,0] op_sel_hi:[0,0,0]", FMT_);      \
  else if constexpr (J == 2) MXL_TILE_MFMA("op_sel_hi:[1,1,0]", FMT_);                     \
  else MXL_TILE_MFMA("op_sel:[1,1,0] op_sel_hi:[1,1,0]", FMT_)
  if constexpr (FMT == kE4M3) { MXL_TILE_MFMA_J(""); }
  else if constexpr (FMT == kE2M3) { MXL_TILE_MFMA_J(" cbsz:2"); }
  else { MXL_TILE_MFMA_J(" cbsz:3"); }
#undef MXL_TILE_MFMA_J
#undef MXL_TILE_MFMA
}

// An accumulator's values, read where they are used (left to the compiler, all of them are
// copied to vector registers at the end of the loop, more than there are)
__device__ __forceinline__ v4f tile_values(const v4f& c) {
  v4f v;
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    float x;
    asm volatile("v_accvgpr_read_b32 %0, %1" : "=v"(x) : "a"(c[e]));
    v[e] = x;
  }
  return v;
}

template <int MTW, int NTW>
struct TileShape {
  static constexpr int BM = 32 * MTW, BN = 32 * NTW;  // workgroup tile
  static constexpr int AU = MTW * 2048, BU = NTW * 2048;  // bytes of an A / B unit
  static constexpr int CA = MTW / 2, CB = NTW / 2;    // copies per wave of a unit (1 KiB each)
  static constexpr int HALF = CA + CB;                // copies per wave of half a stage (one A and one B unit)
};

// What a workgroup computes: rows row0 .. row_hi - 1 (at most BM of them stored) by n-block
// nb, super-tiles kb .. ke - 1.  part: instead of output elements the tile's fp32 partials as
// one block in MFMA fragment order: fragment f = m-tile * (BN / 16) + n-tile is 64 lanes x 4
// floats, lane (q, r) holding columns 4 q .. 4 q + 3 of row r.
struct TileWork {
  int row0, row_hi, nb, kb, ke;
  const uint8_t* w;
  const uint8_t* sw;
  float* part;
};

// LDS of a tile, from its base: the scale slots of two super-tiles (MX: the rows' E8M0 and the
// n-tiles' tiled E8M0 dwords; block-FP8: the rows' fp32 scales [4][BM] and the weight block
// scales of the K range), then `depth` stages of the four units A0, A1, B0, B1.
template <int MTW, int NTW, bool BLOCK>
struct TileLds {
  using S = TileShape<MTW, NTW>;
  static constexpr int SA = 0;
  static constexpr int SB = 2 * S::BM * 16;
  static constexpr int RING = SB + (BLOCK ? (S::BN + 127) / 128 * kWideBlockStages * 4 : 2 * S::BN * 16);
  static constexpr int STAGE = 2 * S::AU + 2 * S::BU;
  static constexpr int bytes(int depth) { return RING + depth * STAGE; }
};

// a_row(row): the activation row of output row `row` (rows past the last: any valid one)
template <int FMT, int MTW, int NTW, bool BLOCK, int DEPTH, class Row>
__device__ __forceinline__ void tile_gemm(const GemmParams& p, const TileWork& w, uint8_t* lds, Row&& a_row) {
  static_assert(!BLOCK || FMT == kE4M3, "block-FP8 weights are E4M3");
  using S = TileShape<MTW, NTW>;
  using L = TileLds<MTW, NTW, BLOCK>;
  constexpr int MH = MTW / 2, NH = NTW / 2, CH = FmtTraits<FMT>::CH;
  // A stage's copies take the slots of the stage DEPTH before it in the order those fall free.
  // At an odd depth that stage reads its B units in the other order, so the B unit this stage
  // needs first is copied second, and the barrier that hands it over waits for CB copies more.
  constexpr int ODD = DEPTH & 1 ? S::CB : 0;
  const int t = threadIdx.x, lane = t & 63;
  const int wv = __builtin_amdgcn_readfirstlane(t >> 6);
  const int wm = wv >> 1, wn = wv & 1;
  const int r = lane & 15, q = lane >> 4;

  // stage and tile indices in 32 bits (the host bounds the operands below 4 GiB)
  const int T = (int)(p.K / 128), KT = (int)p.KT, ntiles = (int)((p.N + 15) / 16), kb = w.kb, ke = w.ke;
  // stages 4 kb .. te - 1; an odd count runs one more (end), whose weights (past K) are zero
  const int te = 4 * ke < T ? 4 * ke : T, end = (te + 1) & ~1;
  const int nt_base = w.nb * (S::BN / 16);

  // copy sources.  A unit h: chunk c = CA wv + u holds rows 8 (c % 2) .. + 7 of the unit's
  // m-tile e = c / 2 (wave row e / MH, its m-tile h MH + e % MH); rows past M re-read the last
  uint32_t a_off[2][S::CA];
#pragma unroll
  for (int h = 0; h < 2; ++h)
#pragma unroll
    for (int u = 0; u < S::CA; ++u) {
      const int c = S::CA * wv + u, e = c >> 1, cr = 8 * (c & 1) + (lane >> 3);
      const int row = a_row(w.row0 + ((e / MH) * MTW + h * MH + e % MH) * 16 + cr);
      a_off[h][u] = (uint32_t)row * (uint32_t)p.lda + 16 * ((lane & 7) ^ tile_swz(cr));
    }
  // B unit h: chunk c = CB wv + u is chunk c % 2 of the unit's n-tile e = c / 2
  const uint8_t* b_src[2][(S::CB + 1) / 2];
#pragma unroll
  for (int h = 0; h < 2; ++h)
#pragma unroll
    for (int u = 0; u < S::CB; u += 2) {
      const int e = (S::CB * wv + u) >> 1;
      int nt = nt_base + (e / NH) * NTW + h * NH + e % NH;
      nt = nt < ntiles ? nt : ntiles - 1;
      b_src[h][u / 2] = w.w + (int64_t)nt * KT * (CH * 1024) + (S::CB == 1 ? (wv & 1) * 1024 : 0);
    }
  const uint32_t lane16 = (uint32_t)lane * 16;
  const uint32_t lds_a = tile_lds(lds + L::RING) + S::CA * wv * 1024;
  const uint32_t lds_b = tile_lds(lds + L::RING) + 2 * S::AU + S::CB * wv * 1024;
  // copies of stage tt into the slot at `slot`
  auto copy_a = [&](int h, int u, int tt, int slot) {
    const int tc = tt < te ? tt : te - 1;  // an odd count's last stage: a valid one again
    tile_copy16(p.a + (uint32_t)tc * 128, a_off[h][u], lds_a + slot + h * S::AU + u * 1024);
  };
  auto copy_b = [&](int h, int u, int tt, int slot) {
    const int j = tt & 3, c0 = FMT == kE4M3 ? 2 * j : (3 * j) >> 1;
    tile_copy16(b_src[h][u >> 1] + (uint32_t)((tt >> 2) * CH + c0 + (u & 1)) * 1024, lane16,
                lds_b + slot + h * S::BU + u * 1024);
  };
  // MX: scales of super-tile kt, 64 rows (16 bytes each) and four n-tiles per wave (where the
  // tile has fewer, several waves copy the same).  A row's window of a part super-tile ends
  // with the row.  Swizzled scales, and rows shorter than a window: dword by dword, 16 rows a
  // copy, clamped to the last slice.  Block-FP8: the four groups' fp32 scales of the rows, one
  // group per wave.
  const bool dwords = !BLOCK && (p.sa_swz || p.K < kTileK);
  const uint32_t srow = (uint32_t)(p.K / 32);
  const int swa = wv % (S::BM / 64), swb = wv % (S::BN / 64);
  uint32_t sa_off[BLOCK ? S::BM / 64 : 1];
  if constexpr (BLOCK) {
#pragma unroll
    for (int c = 0; c < S::BM / 64; ++c) sa_off[c] = (uint32_t)a_row(w.row0 + 64 * c + lane) * 4;
  } else {
    sa_off[0] = (uint32_t)a_row(w.row0 + 64 * swa + lane) * srow;
  }
  int snt = nt_base + 4 * swb + (lane >> 4);
  snt = snt < ntiles ? snt : ntiles - 1;
  const uint32_t sb_off = (uint32_t)snt * (uint32_t)KT * 256 + 16 * (lane & 15);
  const uint32_t lds_sa = tile_lds(lds + L::SA) + (BLOCK ? wv * S::BM * 4 : 64 * swa * 16);
  const uint32_t lds_sb = tile_lds(lds + L::SB) + 4 * swb * 256;
  auto copy_scales = [&](int kt) {
    const int st = kt & 1;
    const int kc = kt < ke ? kt : ke - 1;
    if constexpr (BLOCK) {
      const int g = 4 * kc + wv < T ? 4 * kc + wv : T - 1;
#pragma unroll
      for (int c = 0; c < S::BM / 64; ++c)
        tile_copy4(static_cast<const uint8_t*>(p.sa) + (int64_t)g * p.M * 4, sa_off[c],
                   lds_sa + st * (S::BM * 16) + 256 * c);
    } else {
      if (dwords) {
        const int slice = 4 * kc + (lane & 3) < T ? 4 * kc + (lane & 3) : T - 1;
#pragma unroll
        for (int u = 0; u < S::BM / 64; ++u) {
          const int c = wv + 4 * u;
          tile_copy4(static_cast<const uint8_t*>(p.sa),
                     (uint32_t)(sa_row_offset(p, a_row(w.row0 + 16 * c + (lane >> 2))) + slice * (int)p.sa_ss),
                     tile_lds(lds + L::SA) + st * (S::BM * 16) + 256 * c);
        }
      } else {
        const uint32_t win = 16 * kc + 16 <= (int)srow ? 16 * kc : srow - 16;
        tile_copy16(static_cast<const uint8_t*>(p.sa) + win, sa_off[0], lds_sa + st * (S::BM * 16));
      }
      tile_copy16(w.sw + (uint32_t)kc * 256, sb_off, lds_sb + st * (S::BN * 16));
    }
  };
  const int tb = 4 * kb;
  if constexpr (BLOCK) {
    // the weight block scales of the split's stages, one LDS row per 128 columns (read in the
    // loop from global memory they would be compiler-counted loads, whose waits drain the copies)
#pragma unroll
    for (int c = 0; c < (S::BN + 127) / 128; ++c) {
      const int64_t blocks = (p.N + 127) / 128, want = (int64_t)w.nb * S::BN / 128 + c;
      const uint8_t* src = w.sw + ((want < blocks ? want : blocks - 1) * T + tb) * 4;
      for (int k = 64 * wv; k < te - tb; k += 256) {
        const int at = k + lane < te - tb ? k + lane : te - tb - 1;
        tile_copy4(src, (uint32_t)at * 4, tile_lds(lds + L::SB) + (c * kWideBlockStages + k) * 4);
      }
    }
  }

  v4f acc[MTW][NTW];
#pragma unroll
  for (int i = 0; i < MTW; ++i)
#pragma unroll
    for (int n = 0; n < NTW; ++n) acc[i][n] = v4f{0.f, 0.f, 0.f, 0.f};
  v8i a[2][MH];
  typename TileB<FMT>::type b[2][NH];
  uint32_t sa[MTW], sb[NTW];         // MX: packed E8M0 bytes of the super-tile's slices
  float fa[BLOCK ? MTW : 1][4], fb[4];  // block-FP8: the super-tile's activation and weight scales

  // fragment reads: two LDS reads each
  const int sw = tile_swz(r);
  const int ra = wm * MH * 2048 + (r >> 3) * 1024 + (r & 7) * 128;
  const int ra_lo = ra + 16 * (q ^ sw), ra_hi = ra + 16 * ((q + 4) ^ sw);
  const int rb = wn * NH * 2048 + lane * 16;
  auto read_a = [&](int h, int i, int half, int slot) {  // K 16 q .. (half 0) or 64 + 16 q .. (half 1)
    const uint8_t* src = lds + L::RING + slot + (half ? ra_hi : ra_lo) + h * S::AU + i * 2048;
    const uint4 v = *reinterpret_cast<const uint4*>(src);
    a[h][i][4 * half] = (int)v.x; a[h][i][4 * half + 1] = (int)v.y;
    a[h][i][4 * half + 2] = (int)v.z; a[h][i][4 * half + 3] = (int)v.w;
  };
  auto read_b = [&](int h, int n, int half, int slot, int odd) {  // odd: the parity of the stage's slice
    const uint8_t* src = lds + L::RING + 2 * S::AU + slot + rb + h * S::BU + n * 2048;
    auto& x = b[h][n];
    if constexpr (FMT == kE4M3) {
      const uint4 v = *reinterpret_cast<const uint4*>(src + 1024 * half);
      x[4 * half] = (int)v.x; x[4 * half + 1] = (int)v.y; x[4 * half + 2] = (int)v.z; x[4 * half + 3] = (int)v.w;
    } else if (!odd) {  // even slice: the first chunk and 8 bytes of the second
      if (half == 0) {
        const uint4 v = *reinterpret_cast<const uint4*>(src);
        x[0] = (int)v.x; x[1] = (int)v.y; x[2] = (int)v.z; x[3] = (int)v.w;
      } else {
        const uint2 v = *reinterpret_cast<const uint2*>(src + 1024);
        x[4] = (int)v.x; x[5] = (int)v.y;
      }
    } else {
      if (half == 0) {
        const uint2 v = *reinterpret_cast<const uint2*>(src + 8);
        x[0] = (int)v.x; x[1] = (int)v.y;
      } else {
        const uint4 v = *reinterpret_cast<const uint4*>(src + 1024);
        x[2] = (int)v.x; x[3] = (int)v.y; x[4] = (int)v.z; x[5] = (int)v.w;
      }
    }
  };
  // the lane's E8M0 bytes of a super-tile: byte j of sa[i] is block 4 j + q of its row
  const uint32_t sel_lo = 0x0c0c0400u + 0x0101u * q, sel_hi = 0x04000c0cu + 0x01010000u * q;
  auto read_scales = [&](int kt) {
    const int st = kt & 1;
    if constexpr (BLOCK) {
#pragma unroll
      for (int i = 0; i < MTW; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j)
          fa[i][j] = *reinterpret_cast<const float*>(lds + L::SA + st * (S::BM * 16) +
                                                     (j * S::BM + (wm * MTW + i) * 16 + r) * 4);
      const v4f f = *reinterpret_cast<const v4f*>(lds + L::SB +
                                                  ((S::BN > 128 ? wn : 0) * kWideBlockStages + 4 * kt - tb) * 4);
#pragma unroll
      for (int j = 0; j < 4; ++j) fb[j] = f[j];
      if (4 * kt + 4 > T) {  // the stage past an odd count adds 0 * 0, whatever the last scales are
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          fb[j] = 4 * kt + j < T ? fb[j] : 0.0f;
#pragma unroll
          for (int i = 0; i < MTW; ++i) fa[i][j] = 4 * kt + j < T ? fa[i][j] : 0.0f;
        }
      }
    } else {
      // a part super-tile's window ends with the row: its first byte moves to byte 0
      const int shift = 4 * kt + 4 <= T || dwords ? 0 : 8 * (4 * kt + 4 - T);
#pragma unroll
      for (int i = 0; i < MTW; ++i) {
        const uint4 x = *reinterpret_cast<const uint4*>(lds + L::SA + st * (S::BM * 16) + ((wm * MTW + i) * 16 + r) * 16);
        sa[i] = (__builtin_amdgcn_perm(x.y, x.x, sel_lo) | __builtin_amdgcn_perm(x.w, x.z, sel_hi)) >> shift;
      }
#pragma unroll
      for (int n = 0; n < NTW; ++n)
        sb[n] = *reinterpret_cast<const uint32_t*>(lds + L::SB + st * (S::BN * 16) + (wn * NTW + n) * 256 + lane * 4);
    }
  };

  // Stage tt (slice J of its pair) from the slot at `cur`, the next stage's at `nxt`: four
  // quadrants of Q MFMAs, after each MFMA its share of the reads of the next unit and of the
  // copies of DEPTH stages ahead (into the slots that this stage frees).  LEFT: the stages left,
  // this one included, at the end (0: more than four); then copies would lie past it, and fewer
  // half-stages of copies may stay in flight at a barrier (those after the units it hands over).
  auto stage = [&](auto J, auto LEFT, int tt, int cur, int nxt) {
    constexpr int st = decltype(J)::value & 1, x = st, y = 1 - st, left = decltype(LEFT)::value;
    constexpr bool ahead = left == 0 || left > DEPTH;
    constexpr int full = 2 * DEPTH - 2;
    constexpr int Q = MH * NH;
    v4f raw[3];
    float f[BLOCK ? MTW : 1];
    if constexpr (BLOCK) {
#pragma unroll
      for (int i = 0; i < MTW; ++i) f[i] = fa[i][st] * fb[st];
    }
    // block-FP8: acc = fma(raw, sa sb, acc) of the stage's g-th MFMA, two MFMAs after it
    auto fold = [&](int g) {
      const int s = g / Q, k = g % Q, i = (s >> 1) * MH + k / NH, n = (s == 0 || s == 3 ? x : y) * NH + k % NH;
#pragma unroll
      for (int e = 0; e < 4; ++e) acc[i][n][e] = __builtin_fmaf(raw[g % 3][e], f[BLOCK ? i : 0], acc[i][n][e]);
    };
    auto quad = [&](auto QI, auto&& between) {
      constexpr int s = decltype(QI)::value, ah = s >> 1, bh = s == 0 || s == 3 ? x : y;
#pragma unroll
      for (int i = 0; i < MH; ++i)
#pragma unroll
        for (int n = 0; n < NH; ++n) {
          const int k = i * NH + n, g = s * Q + k;
          if constexpr (BLOCK) {
            const v4f z = {0.f, 0.f, 0.f, 0.f};
            raw[g % 3] = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(b[bh][n], a[ah][i], z, kE4M3, kE4M3, 0, 127, 0,
                                                                          127);
            if (g >= 2) fold(g - 2);
          } else {
            tile_mfma<FMT, decltype(J)::value>(acc[ah * MH + i][bh * NH + n], b[bh][n], a[ah][i], sb[bh * NH + n],
                                               sa[ah * MH + i]);
          }
          between(k);
          if constexpr (BLOCK) __builtin_amdgcn_sched_barrier(0);
        }
    };
    // a unit's `total` reads or copies spread over the Q MFMAs: the share of MFMA k
    auto reads_a = [&](int k, int h, int slot) {
      constexpr int R = (2 * MH + Q - 1) / Q;
#pragma unroll
      for (int u = 0; u < R; ++u)
        if (k * R + u < 2 * MH) read_a(h, (k * R + u) >> 1, (k * R + u) & 1, slot);
    };
    auto reads_b = [&](int k, int h, int slot, int odd) {
      constexpr int R = (2 * NH + Q - 1) / Q;
#pragma unroll
      for (int u = 0; u < R; ++u)
        if (k * R + u < 2 * NH) read_b(h, (k * R + u) >> 1, (k * R + u) & 1, slot, odd);
    };
    auto copies_a = [&](int k, int h) {
      if constexpr (!ahead) {
      } else if constexpr (Q >= S::CA) {
        if (k % (Q / S::CA) == Q / S::CA - 1) copy_a(h, k / (Q / S::CA), tt + DEPTH, cur);
      } else {
#pragma unroll
        for (int u = 0; u < S::CA / Q; ++u) copy_a(h, k * (S::CA / Q) + u, tt + DEPTH, cur);
      }
    };
    auto copies_b = [&](int k, int h) {
      if constexpr (!ahead) {
      } else if constexpr (Q >= S::CB) {
        if (k % (Q / S::CB) == Q / S::CB - 1) copy_b(h, k / (Q / S::CB), tt + DEPTH, cur);
      } else {
#pragma unroll
        for (int u = 0; u < S::CB / Q; ++u) copy_b(h, k * (S::CB / Q) + u, tt + DEPTH, cur);
      }
    };
    tile_wait<S::HALF * (left && 2 * left - 2 < full ? 2 * left - 2 : full)>();
    quad(Slice<0>{}, [&](int k) { reads_b(k, y, cur, st); copies_a(k, 0); });
    quad(Slice<1>{}, [&](int k) { reads_a(k, 1, cur); copies_b(k, x); });
    if constexpr (left != 1) tile_wait<S::HALF * (ahead ? full : 2 * left - 3) - ODD>();
    quad(Slice<2>{}, [&](int k) { reads_a(k, 0, nxt); copies_b(k, y); });
    quad(Slice<3>{}, [&](int k) { reads_b(k, y, nxt, 1 - st); copies_a(k, 1); });
    if constexpr (BLOCK) {
      fold(4 * Q - 2);
      fold(4 * Q - 1);
    }
  };

  copy_scales(kb);
  const int count = end - tb;  // stages: an even number
#pragma unroll
  for (int k = 0; k < DEPTH; ++k) {  // units in the order the loop copies them
    if (k >= 2 && k >= count) break;
    const int x = (k + DEPTH) & 1;
#pragma unroll
    for (int u = 0; u < S::CA; ++u) copy_a(0, u, tb + k, k * L::STAGE);
#pragma unroll
    for (int u = 0; u < S::CB; ++u) copy_b(x, u, tb + k, k * L::STAGE);
#pragma unroll
    for (int u = 0; u < S::CB; ++u) copy_b(1 - x, u, tb + k, k * L::STAGE);
#pragma unroll
    for (int u = 0; u < S::CA; ++u) copy_a(1, u, tb + k, k * L::STAGE);
  }
  if (DEPTH > 2 && count == 2) tile_wait<S::HALF * 3 - ODD>();
  else tile_wait<S::HALF * (2 * DEPTH - 1) - ODD>();
#pragma unroll
  for (int i = 0; i < MH; ++i) { read_a(0, i, 0, 0); read_a(0, i, 1, 0); }
#pragma unroll
  for (int n = 0; n < NH; ++n) { read_b(0, n, 0, 0, 0); read_b(0, n, 1, 0, 0); }

  // two stages per iteration, byte pairs 0, 1 then 2, 3 of the packed scales
  int cur = 0;  // the slot of the pair's first stage
  auto pair = [&](auto LEFT, int pr) {  // LEFT: the stages left at the pair's first, 0 for many
    const int kt = pr >> 1;
    if ((pr & 1) == 0) {
      if (kt + 1 < ke) copy_scales(kt + 1);
      read_scales(kt);  // landed: the copies of the stages before this one were issued after them
    } else if constexpr (BLOCK) {
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        fb[j] = fb[j + 2];
#pragma unroll
        for (int i = 0; i < MTW; ++i) fa[i][j] = fa[i][j + 2];
      }
    } else {
#pragma unroll
      for (int i = 0; i < MTW; ++i) sa[i] >>= 16;
#pragma unroll
      for (int n = 0; n < NTW; ++n) sb[n] >>= 16;
    }
    if constexpr (!BLOCK) {  // (the empty statements keep the operands' last writes ahead of the s_nop)
#pragma unroll
      for (int i = 0; i < MTW; ++i)
#pragma unroll
        for (int n = 0; n < NTW; ++n) asm volatile("" : "+a"(acc[i][n]));
#pragma unroll
      for (int i = 0; i < MTW; ++i) asm volatile("" : "+v"(sa[i]));
#pragma unroll
      for (int n = 0; n < NTW; ++n) asm volatile("" : "+v"(sb[n]));
      asm volatile("s_nop 1");
    }
    constexpr int left = decltype(LEFT)::value;
    constexpr int ring = DEPTH * L::STAGE;
    const int one = cur + L::STAGE < ring ? cur + L::STAGE : 0, two = one + L::STAGE < ring ? one + L::STAGE : 0;
    stage(Slice<0>{}, Slice<left>{}, 2 * pr, cur, one);
    stage(Slice<1>{}, Slice<left ? left - 1 : 0>{}, 2 * pr + 1, one, two);
    // 64 x 64 tiles: the compiler moves the accumulators after the loop, 17 states after the last MFMA whose
    // result takes 20
    if constexpr (!BLOCK && MTW * NTW == 4) asm volatile("s_nop 2");
    cur = two;
  };
  const int last = end >> 1;  // pairs 2 kb .. last - 1; the copies end in the final one or two
  int pr = 2 * kb;
  for (; pr + (DEPTH > 2 ? 2 : 1) < last; ++pr) pair(Slice<0>{}, pr);
  if (DEPTH > 2 && pr + 1 < last) pair(Slice<4>{}, pr++);
  pair(Slice<2>{}, pr);

  auto values = [&](int i, int n) -> v4f {
    if constexpr (BLOCK) return acc[i][n];
    else return tile_values(acc[i][n]);
  };
  if constexpr (!BLOCK) asm volatile("s_nop 15\n\ts_nop 15" ::: "memory");  // the last MFMAs' results
  // lane (q, r): columns 4 q .. 4 q + 3 of row r of every 16 x 16 tile
  if (w.part) {
#pragma unroll
    for (int i = 0; i < MTW; ++i)
#pragma unroll
      for (int n = 0; n < NTW; ++n) {
        const int f = (wm * MTW + i) * (S::BN / 16) + wn * NTW + n;
        *reinterpret_cast<v4f*>(w.part + (f * 64 + lane) * 4) = values(i, n);
        __builtin_amdgcn_sched_barrier(0);
      }
  } else if (p.N % 4 == 0 && p.ldc % 4 == 0 && p.ldc < (1 << 22) && ((uintptr_t)p.out & 7) == 0 && !p.out_f16 &&
             p.alpha == 1.0f) {
    // Buffer stores drop what lies past the last row (the buffer ends with it) or column (an
    // offset past the buffer), so the accumulators leave without a branch each.
    typedef unsigned int u2 __attribute__((ext_vector_type(2)));
    uint16_t* const base = p.out + (int64_t)w.row0 * p.ldc;
    const int rows = w.row_hi - w.row0 < S::BM ? w.row_hi - w.row0 : S::BM, ld = (int)p.ldc;
    const __amdgpu_buffer_rsrc_t rs =
        __builtin_amdgcn_make_buffer_rsrc((void*)base, (short)0, ((rows - 1) * ld + (int)p.N) * 2, 0x00020000);
    const int r0 = wm * MTW * 16 + r, c0 = w.nb * S::BN + wn * NTW * 16 + 4 * q;
    // two bf16 of two fp32 (NaNs quiet)
    auto pack = [](float x, float y) -> uint32_t {
      uint32_t d = cvt_pk_bf16(x, y);
      d = x != x ? (d & 0xFFFF0000u) | 0x7FC0u : d;
      return y != y ? (d & 0x0000FFFFu) | 0x7FC00000u : d;
    };
    // BIAS: one is added to the rounded output (MXFP8 2048 x 18432 x 2560 135 us with a pass of its
    // own, 104 here, 222 through the LDS below)
    auto store = [&](auto BIAS) {
      u2 bias[NTW];
      if constexpr (decltype(BIAS)::value) {
#pragma unroll
        for (int n = 0; n < NTW; ++n) {
          const uint16_t* const src = p.bias + (c0 + 16 * n < (int)p.N ? c0 + 16 * n : 0);
#pragma unroll
          for (int e = 0; e < 2; ++e) bias[n][e] = src[2 * e] | (uint32_t)src[2 * e + 1] << 16;
        }
      }
#pragma unroll
      for (int i = 0; i < MTW; ++i)
#pragma unroll
        for (int n = 0; n < NTW; ++n) {
          const v4f v = values(i, n);
          u2 h;
#pragma unroll
          for (int e = 0; e < 2; ++e) {
            h[e] = pack(v[2 * e], v[2 * e + 1]);
            if constexpr (decltype(BIAS)::value)
              h[e] = pack(u2f(h[e] << 16) + u2f(bias[n][e] << 16),
                          u2f(h[e] & 0xFFFF0000u) + u2f(bias[n][e] & 0xFFFF0000u));
          }
          const uint32_t off = c0 + 16 * n < (int)p.N ? (uint32_t)((r0 + 16 * i) * ld + c0 + 16 * n) * 2 : 0xFFFFFFF0u;
          __builtin_amdgcn_raw_buffer_store_b64(h, rs, (int)off, 0, 0);
          __builtin_amdgcn_sched_barrier(0);
        }
    };
    if (p.bias) store(Slice<1>{});
    else store(Slice<0>{});
  } else {
    // other output formats and alignments: 16 rows at a time through the wave's own
    // part of the ring, once every wave is past its last read of it
    constexpr int TW = 16 * NTW;
    static_assert(4 * 16 * TW * 4 <= 2 * L::STAGE, "the staged rows fit the ring");
    float* const stage_out = reinterpret_cast<float*>(lds + L::RING) + wv * 16 * TW;
    tile_wait<0>();
#pragma unroll
    for (int i = 0; i < MTW; ++i) {
#pragma unroll
      for (int n = 0; n < NTW; ++n) *reinterpret_cast<v4f*>(stage_out + r * TW + 16 * n + 4 * q) = values(i, n);
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
#pragma unroll 1
      for (int c = lane; c < 16 * TW; c += 64) {
        const int64_t row = w.row0 + (wm * MTW + i) * 16 + c / TW, col = (int64_t)w.nb * S::BN + wn * TW + c % TW;
        const float v = stage_out[c];
        if (row < w.row_hi && col < p.N) p.out[row * p.ldc + col] = out_bits(p, v, col);
      }
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    }
  }
}

}  // namespace mxl
