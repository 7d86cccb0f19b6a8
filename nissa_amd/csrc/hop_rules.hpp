// Storage kinds of spinors and links, and the rules by which a twisted-mass hop picks its
// kernel and cache policy.  Free of HIP: a host compiler builds the rules as go() uses them.
#pragma once

#include <cstdint>

namespace nq {

// ---------------------------------------------------------------- storage kinds
enum SpPrec { SP_F64 = 0, SP_F32 = 1, SP_F16 = 2 };
enum LkPrec { LK_F64_18 = 0, LK_F32_18 = 1, LK_F32_12 = 2, LK_F16_12 = 3, LK_F64_12 = 4 };
// complex elements stored per link (12-real: rows 0 and 1) and bytes per element
constexpr int lk_nc(int lk) { return (lk == LK_F64_18 || lk == LK_F32_18) ? 9 : 6; }
constexpr int lk_eb(int lk) { return (lk == LK_F64_18 || lk == LK_F64_12) ? 16 : (lk == LK_F16_12 ? 4 : 8); }

// Whether the links and the data used once are accessed with the default cache policy,
// to be found in the 256 MB memory-side cache by the next hop, instead of streamed past
// it: when the links of both parities (and the clover blocks of K) and the input and
// output spinors take at most 224 MB (150 MB for several right-hand sides, whose other
// vectors grow with them).  Measured, default against streamed, whole solves
// (links of both parities): 123 MB (FP16 inner, 20^3x40) 7.41 against 8.23 ms, 127 MB
// (FP16 links, 24^3x48) 11.6 / 12.7, 151 MB (FP64, 16^3x32) 7.56 / 8.03, 184 MB (FP32,
// 20^3x40) 9.35 / 10.2; above it 236 MB (FP16 links, 28^3x56) 22.0 / 21.2, 255 MB (FP16
// inner, 24^3x48) 14.5 / 14.1, 369 MB (FP64, 20^3x40) 19.9 / 19.0, 805 MB (FP16 inner,
// 32^3x64) 41.2 / 37.4.  Twelve FP16 right-hand sides: 50 MB of links 21.8 / 22.1, 123 MB
// (and 200 MB of spinors) 56.6 / 54.6, 255 MB 114.6 / 108.6; five at 46x16x22x20, 124 and
// 84 MB, 26.4 / 25.9.
inline bool links_stay(int64_t Vh, int sp, int lk, int nr, bool clover)
{
  const int eb = sp == SP_F64 ? 16 : (sp == SP_F32 ? 8 : 4);
  double site = 2.0 * 8 * lk_nc(lk) * lk_eb(lk) + 2.0 * 12 * eb * nr;
  if (clover) site += (72 + 36) * eb;
  return site * (double)Vh <= (nr > 1 ? 150.0 : 224.0) * 1048576;
}

// Neighbours staged in LDS (k_tm_hop_lds) for one right-hand side: FP64 always (4 % at
// 32^3x64), the sloppy precisions when the links are streamed: unstaged against staged,
// FP32 54.4 / 49.8 us at 24^3x48 and 139 / 132 at 32^3x64; FP16 34.1 / 33.4 and 91 / 86;
// FP16 links at 32^3x64 66.5 / 63.5.  With the links in the memory-side cache the staging
// round trip is not paid back: 16^3x32 FP32 10.7 / 12.0 us, FP16 9.4 / 10.1, FP16 links
// 9.1 / 9.7; 24^3x48, FP16 links 24.1 / 25.6.
inline bool use_lds(int sp, bool keep) { return sp == SP_F64 || !keep; }

// Hops of one right-hand side split the directions over the wavefronts of a workgroup
// (k_tm_hop_split and k_tm_hop_split_any) on lattices below a number of sites per parity.
// Plain FP64 below 2^18, where the persistent kernel does not fill its slots twice; one
// thread per site / split: hop on 8^4 10.3 / 4.6 us, 12x6x10x14 14.5 / 4.7, 24x12^3 16.6 /
// 7.4, 16^3x32 20.2 / 18.6, 20^3x40 55.0 / 48.6; above, 24^3x48 98 / 103, 28^3x56 177 / 190.
// The others finish a site in one wavefront of four and lose sooner.  Sloppy precisions
// below 2^17: FP16 inner solves at 8^3x16 3.22 / 2.35 ms, 24x12^3 3.52 / 2.65, 16^3x32 4.42 /
// 3.95 (FP32 4.49 / 4.31), 20^3x40 6.95 / 6.98.  Clover blocks, FP16 and FP32 below 2^15:
// 24x12^3 3.89 / 3.06 ms, 16^3x32 4.92 / 5.21; FP64 below 2^13: 8^3x16 3.76 / 3.18 ms,
// 24x12^3 4.67 / 5.20.
inline bool use_split(int64_t Vh, int sp, bool plain64, bool clover)
{
  const int bits = plain64 ? 18 : (!clover ? 17 : (sp == SP_F64 ? 13 : 15));
  return Vh < (int64_t(1) << bits);
}

// Neighbours staged in LDS in the register-blocked kernel, as far as the LDS holds two
// workgroups or more (FP16 any RB, FP32 up to two, FP64 one right-hand side per wavefront).
// The batched hop is bound by the L2->L1 path: twelve right-hand sides at 24^3x48, FP64
// 825 -> 713 us, FP32 400 -> 308.  Where the blocks of all right-hand sides do not give
// every CU more than one, the staging round trip only adds latency.  FP32 solves, not
// staged / staged: 8^3x16, 2 sources 4.24 / 4.51 ms, 12 sources 6.30 / 6.68; 20x12^3, 2
// sources 5.09 / 5.41, 5 sources 6.70 / 6.62, 8 sources 9.01 / 8.28; 32x12x14x12, 2 sources
// 5.54 / 5.72, 3 sources 6.46 / 6.49; 20x16^3, 2 sources 6.26 / 6.01; 16x10x12^2, 5 sources
// 5.98 / 6.36, 8 sources 7.08 / 7.31, 12 sources 9.58 / 8.97.  The staging is a template
// parameter: as a branch it cost the launches that skip it 1.2 us of 10, and the FP16 tail
// a wavefront per SIMD (five sources at 20^3x40: 61 -> 70 us).
constexpr bool batch_stages(int sp, int rb) { return sp == SP_F16 || (sp == SP_F32 && rb <= 2) || (sp == SP_F64 && rb == 1); }
inline bool stage_batch(int64_t Vh, int sp, int rb, int nr, int ncu)
{
  return batch_stages(sp, rb) && (Vh + 255) / 256 * nr > ncu;
}

// Kernel and cache policy of a hop that is not register-blocked.  xp: precision of the
// other fields of the epilogue's tail; per_rhs: coefficients per right-hand side (a batch,
// whose kernel does not depend on its size); lds: staging allowed.  keep: the default cache
// policy (links_stay), for every kernel: the FP64 residual hop of a mixed solve too, whose
// links would take the sloppy links' place in the memory-side cache (FP16, FP16 links and
// FP32 inner iterations at 32x20^3, 128000 sites per parity, default / streamed there:
// 6.36 / 6.34, 5.85 / 5.85, 7.30 / 7.27 ms; equal where the residual hop's links fit).
enum HopKernel { HOP_PLAIN = 0, HOP_LDS = 1, HOP_SPLIT = 2 };
struct HopRoute {
  HopKernel kernel;
  bool keep;
};
inline HopRoute hop_route(int64_t Vh, int sp, int lk, int xp, bool clover, int nr, bool per_rhs, bool lds)
{
  HopRoute r = {HOP_PLAIN, links_stay(Vh, sp, lk, nr, clover)};
  const bool plain64 = sp == SP_F64 && xp == SP_F64 && !clover;
  if (nr != 1) return r;
  if (!per_rhs && use_split(Vh, sp, plain64, clover)) r.kernel = HOP_SPLIT;
  else if (lds && use_lds(sp, r.keep)) r.kernel = HOP_LDS;
  return r;
}

// Whether HOP_LDS can come with keep: the sloppy precisions stage streamed links only, and a
// plain FP64 hop that is not split (2^18 sites) exceeds the 224 MB.  Not so the clover hops
// and, in a batch, the residual (mode 3).
constexpr bool hop_lds_keeps(int sp, int mode, bool clover) { return sp == SP_F64 && (mode == 3 || clover); }

// Right-hand sides per wavefront of the staggered hops for nr > 1: 6 for FP32 batches of
// five or more, else 4, and fewer on a lattice whose 256-site blocks then give less than two
// workgroups per CU.  Multi-shift CG, with 4 or 6 -> with the block taken: 16^3x32, 4
// sources, 10 shifts, FP32 51.5 -> 46.9 ms, FP64 42.6 -> 39.1; 26x14^3, 3 x 9, FP32 35.6 ->
// 30.5; 16x8^3, 4 x 12, 33.1 -> 24.4; 20x10^3, 2 x 8, FP64 17.2 -> 14.5.  20^3x40, 4 x 10,
// FP64 keeps 4: 102.5 (2: 101.1, 1: 126.5).
// One per wavefront re-reads the links for every source, and pays only while the blocks of
// all sources leave the card that empty: one block (FP64) or two (FP32) per CU.  RB = 1 / 2:
// FP64 28x12^2x14, 2 sources 17.6 / 19.0 ms, 3 sources 23.7 / 20.3; 20x16^3, 2 sources 16.5 /
// 14.0, 4 sources 25.7 / 20.1; 24x20^3, 2 sources 31.8 / 26.3; FP32 20x16^3, 2 sources 19.8 /
// 21.0; 26x16^3, 4 sources 37.8 / 34.4; 24x20^3, 2 sources 28.6 / 27.2.
inline int st_block(int64_t Vh, int nr, int sp, int ncu)
{
  const int64_t nblk = (Vh + 255) / 256, alone = (sp == SP_F64 ? 1 : 2) * ncu;
  int v = sp == SP_F32 && nr >= 5 ? 6 : 4;
  while (v > 1 && nblk * ((nr + v - 1) / v) < 2 * ncu && (v > 2 || nblk * nr <= alone)) v = v > 4 ? 4 : v / 2;
  return v;
}

// Rows of a z tile of the site order (halved until it divides the extent).  Two, which with
// the 4 x 2 patch make 256 consecutive sites of a 64-slice t tile a 2 x 2 x 2 cell of rows.
// Eight below 2^16 sites per parity, where a wavefront covers many rows: its x and y
// neighbours are then all inside the workgroup or all outside it, and a load is not split in
// two by the branch (two / eight rows: two FP32 sources on 8^4 4.26 / 3.93 ms, three at
// 24x12^2x16 6.07 / 5.75; FP64 shifts, one source, 16x6^2x8 13.3 / 12.8; 16^3x32, three FP32
// sources, 9.30 / 9.66).  Four where the t extent is no multiple of eight and the rows cut
// across wavefronts (two / four: two FP16 sources at 30x24^3 15.8 / 15.5 ms, six 36.6 / 35.6;
// FP64 at 22x26x28^2 22.5 / 22.2; 24^4 and 32x20^3 equal or worse).
inline int z_tile(int T, int64_t Vh) { return Vh < (int64_t(1) << 16) ? 8 : (T % 8 ? 4 : 2); }

}  // namespace nq
