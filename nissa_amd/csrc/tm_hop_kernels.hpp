// Twisted-mass Wilson hopping term of one parity with fused epilogues, for gfx950.
//
// Reference: tmn2Deo_or_tmn2Doe_eos (src/dirac_operators/tmD_eoprec/
// dirac_operator_tmD_eoprec_portable.hpp:36-169):
//   out(x) = sum_mu (1 - g_mu) U_mu(x) in(x+mu) + (1 + g_mu) U_mu(x-mu)^+ in(x-mu)
// in nissa's gamma basis (src/new_types/dirac.cpp:43-58).  The spin projections
// and the way the two projected colour vectors are scattered back onto the four
// spins are fixed by that basis, so the per-direction table below necessarily
// matches the reference's (same algebra, written for our accumulators).
//
// One thread per output site; links are streamed from the per-output-parity
// slot arrays (backward links pre-daggered at upload), neighbour spinors are
// gathered from the opposite-parity SoA field (L2/MALL-resident).  The epilogue
// applies the site-local pieces of the eo operator in registers:
//   out_h = c1_h hop + c2_h aux + c3_h aux2    (h = upper/lower spin pair)
// which covers tmn2D, inv_tmDee(hop), g5(Doo in - hop/4), g5(eta + hop/2),
// Dee^-1(eta + hop/2), and Q = g5 D on each parity; mode 2 fuses the CG update
// x += alpha p, r -= alpha s and |r|^2; mode 3 writes a residual b - A x in FP64
// plus its sloppy copy and |r|^2.

#pragma once

#include <hip/hip_ext.h>

#include <algorithm>
#include <cstdlib>
#include <string>
#include "clover_block.hpp"

namespace nq {

// Hop launches: with the ledger on (ctx->hop_ev set by prof_begin_ext) the launch
// records the kernel's own start and end, so that the ledger's time per launch is
// the kernel's, as in a profiler's kernel trace, without the dispatch gap that two
// stream events around the launch would add.
#define NQ_HOP_LAUNCH(KERNEL, GRID, BLOCK, ...)                                                          \
  do {                                                                                                  \
    if (ctx->hop_ev[0])                                                                                 \
      hipExtLaunchKernelGGL(KERNEL, GRID, BLOCK, 0, ctx->stream, ctx->hop_ev[0], ctx->hop_ev[1], 0, __VA_ARGS__); \
    else                                                                                                \
      hipLaunchKernelGGL(KERNEL, GRID, BLOCK, 0, ctx->stream, __VA_ARGS__);                             \
  } while (0)

template <class R>
struct Half {
  cx<R> h0[3], h1[3];
};

// spin projection of the neighbour spinor for slot (mu, fwd/bwd)
template <class R, int MU, bool FWD>
__device__ __forceinline__ void project(const cx<R> s[12], cx<R> h0[3], cx<R> h1[3])
{
#pragma unroll
  for (int c = 0; c < 3; c++) {
    const cx<R> s0 = s[c], s1 = s[3 + c], s2 = s[6 + c], s3 = s[9 + c];
    if constexpr (FWD) {  // (1 - gamma_mu)
      if constexpr (MU == 0) { h0[c] = s0 + s2; h1[c] = s1 + s3; }
      if constexpr (MU == 1) { h0[c] = iadd(s0, s3); h1[c] = iadd(s1, s2); }
      if constexpr (MU == 2) { h0[c] = s0 + s3; h1[c] = s1 - s2; }
      if constexpr (MU == 3) { h0[c] = iadd(s0, s2); h1[c] = isub(s1, s3); }
    } else {  // (1 + gamma_mu)
      if constexpr (MU == 0) { h0[c] = s0 - s2; h1[c] = s1 - s3; }
      if constexpr (MU == 1) { h0[c] = isub(s0, s3); h1[c] = isub(s1, s2); }
      if constexpr (MU == 2) { h0[c] = s0 - s3; h1[c] = s1 + s2; }
      if constexpr (MU == 3) { h0[c] = isub(s0, s2); h1[c] = iadd(s1, s3); }
    }
  }
}

// Spin projection of an FP16 neighbour straight from its stored halves: every
// component of h0 and h1 is a sum or difference of two halves, formed in FP32 by one
// v_fma_mix_f32 (a * 1 + b on operands widened in the instruction: one rounding, as
// the FP32 add of the widened halves has), and scaled by the site's norm afterwards.
// That takes 24 instructions a slot where widening, scaling and adding took 60; the
// batched hop spends about two thirds of its time on the VALU, on which v_cvt_f32_f16
// runs at half the rate of an FP32 multiply or add (4.4 against 2.6 cycles a wavefront).
// The factor 1 is opaque to the compiler, which would otherwise turn the FMA into
// conversions and an add.
template <int MU, bool FWD>
__device__ __forceinline__ void project_f16(const RawF16& w, float scale, cx<float> h0[3], cx<float> h1[3])
{
  float one;
  asm("v_mov_b32 %0, 1.0" : "=v"(one));
  auto add = [one](float a, float b) { return __builtin_fmaf(a, one, b); };
  auto sub = [one](float a, float b) { return __builtin_fmaf(-b, one, a); };
  auto cadd = [&](cx<float> a, cx<float> b) { return mk<float>(add(a.re, b.re), add(a.im, b.im)); };
  auto csub = [&](cx<float> a, cx<float> b) { return mk<float>(sub(a.re, b.re), sub(a.im, b.im)); };
  auto ciadd = [&](cx<float> a, cx<float> b) { return mk<float>(sub(a.re, b.im), add(a.im, b.re)); };
  auto cisub = [&](cx<float> a, cx<float> b) { return mk<float>(add(a.re, b.im), sub(a.im, b.re)); };
#pragma unroll
  for (int c = 0; c < 3; c++) {
    const cx<float> s0 = w.at(c), s1 = w.at(3 + c), s2 = w.at(6 + c), s3 = w.at(9 + c);
    if constexpr (MU == 0) { h0[c] = FWD ? cadd(s0, s2) : csub(s0, s2); h1[c] = FWD ? cadd(s1, s3) : csub(s1, s3); }
    if constexpr (MU == 1) { h0[c] = FWD ? ciadd(s0, s3) : cisub(s0, s3); h1[c] = FWD ? ciadd(s1, s2) : cisub(s1, s2); }
    if constexpr (MU == 2) { h0[c] = FWD ? cadd(s0, s3) : csub(s0, s3); h1[c] = FWD ? csub(s1, s2) : cadd(s1, s2); }
    if constexpr (MU == 3) { h0[c] = FWD ? ciadd(s0, s2) : cisub(s0, s2); h1[c] = FWD ? cisub(s1, s3) : ciadd(s1, s3); }
    h0[c] = scal(h0[c], scale);
    h1[c] = scal(h1[c], scale);
  }
}

// The projected neighbour n of right-hand side r for slot (MU, FWD), from LDS (staged
// sites [lds_e0, lds_e0 + kStageSites)) or memory.
template <int SP, class R, int MU, bool FWD>
__device__ __forceinline__ void load_projected(const Geo& g, const SpinorView& in, int r, uint32_t n, const char* lds,
                                               uint32_t lds_e0, cx<R> h0[3], cx<R> h1[3])
{
  const uint32_t d = n - lds_e0;
  if constexpr (SP == SP_F16) {
    RawF16 w;
    if (lds && d < (uint32_t)kStageSites) Stage<SP, 12>::get_raw(lds, (int)d, w);
    else w.load(in, g.stride, n, r);
    project_f16<MU, FWD>(w, w.norm, h0, h1);
  } else {
    cx<R> sp[12];
    if (lds && d < (uint32_t)kStageSites) Stage<SP, 12>::get(lds, (int)d, sp);
    else SpAcc<SP, R, 12>::load(in, g.stride, n, sp, r);
    project<R, MU, FWD>(sp, h0, h1);
  }
}

// reconstruct the four spins from the two multiplied half spinors
template <class R, int MU, bool FWD>
__device__ __forceinline__ void scatter(cx<R> o[12], const cx<R> g0[3], const cx<R> g1[3])
{
#pragma unroll
  for (int c = 0; c < 3; c++) {
    o[c] = o[c] + g0[c];
    o[3 + c] = o[3 + c] + g1[c];
    if constexpr (FWD) {
      if constexpr (MU == 0) { o[6 + c] = o[6 + c] + g0[c]; o[9 + c] = o[9 + c] + g1[c]; }
      if constexpr (MU == 1) { o[6 + c] = isub(o[6 + c], g1[c]); o[9 + c] = isub(o[9 + c], g0[c]); }
      if constexpr (MU == 2) { o[6 + c] = o[6 + c] - g1[c]; o[9 + c] = o[9 + c] + g0[c]; }
      if constexpr (MU == 3) { o[6 + c] = isub(o[6 + c], g0[c]); o[9 + c] = iadd(o[9 + c], g1[c]); }
    } else {
      if constexpr (MU == 0) { o[6 + c] = o[6 + c] - g0[c]; o[9 + c] = o[9 + c] - g1[c]; }
      if constexpr (MU == 1) { o[6 + c] = iadd(o[6 + c], g1[c]); o[9 + c] = iadd(o[9 + c], g0[c]); }
      if constexpr (MU == 2) { o[6 + c] = o[6 + c] + g1[c]; o[9 + c] = o[9 + c] - g0[c]; }
      if constexpr (MU == 3) { o[6 + c] = iadd(o[6 + c], g0[c]); o[9 + c] = isub(o[9 + c], g1[c]); }
    }
  }
}

// lds: staged records of sites [lds_e0, lds_e0 + kStageSites) of `in`, or null
template <int SP, int LK, class R, int MU, bool FWD, bool PIN, int CP, bool STAGED>
__device__ __forceinline__ void hop_slot(const Geo& g, const Site& s, uint32_t e, const SpinorView& in, int r,
                                         const void* ub, const double* det, unsigned unit, R anis, bool use_anis,
                                         cx<R> o[12], const char* lds = nullptr, uint32_t lds_e0 = 0)
{
  const uint32_t n = neigh_eo(g, s, MU, FWD);
  constexpr int slot = 2 * MU + (FWD ? 0 : 1);
  // staged: the link's loads first; with the neighbour in LDS or memory (a branch) in
  // front of them they would be issued only after its wait
  cx<R> u[9], h0[3], h1[3];
  if constexpr (STAGED) LkAcc<LK, R, CP>::load_stored(ub, g.stride, slot, e, u);
  load_projected<SP, R, MU, FWD>(g, in, r, n, STAGED ? lds : nullptr, lds_e0, h0, h1);
  if constexpr (!STAGED) LkAcc<LK, R, CP>::load_stored(ub, g.stride, slot, e, u);
  LkAcc<LK, R, CP>::complete(det + 2 * slot, u, lk_eb(LK) < 16 && ((unit >> MU) & 1u));
  cx<R> g0[3], g1[3];
  mat_vec(u, h0, g0);
  mat_vec(u, h1, g1);
  if (MU > 0 && use_anis) {
#pragma unroll
    for (int c = 0; c < 3; c++) { g0[c] = scal(g0[c], anis); g1[c] = scal(g1[c], anis); }
  }
  scatter<R, MU, FWD>(o, g0, g1);
  // Materialise the accumulators before the next group of slots issues its loads:
  // without this the compiler sinks the arithmetic of all eight slots below all
  // their loads and keeps ~400 values live (FP64 spills to scratch).  Groups of
  // four slots keep enough loads in flight per wait (measured best on gfx950).
  if constexpr (PIN) {
#pragma unroll
    for (int k = 0; k < 12; k++) asm volatile("" : "+v"(o[k].re), "+v"(o[k].im));
    asm volatile("" ::: "memory");
  }
}

// The eight slots of one output site, the accumulators pinned after every PK slots
// (PK = 4: two groups of four slots; the persistent FP64 kernel takes PK = 2).  The
// pins order the schedule only; the arithmetic, and so every bit of the result, is
// the same for every PK.
template <int SP, int LK, class R, int PK, int CP, bool STAGED>
__device__ __forceinline__ void hop_site(const Geo& g, const Site& s, uint32_t e, const SpinorView& in, int r,
                                         const void* ub, const double* det, unsigned unit, R anis, bool ua, cx<R> o[12],
                                         const char* lds = nullptr, uint32_t e0 = 0)
{
  hop_slot<SP, LK, R, 0, true, (1 % PK) == 0, CP, STAGED>(g, s, e, in, r, ub, det, unit, anis, ua, o, lds, e0);
  hop_slot<SP, LK, R, 0, false, (2 % PK) == 0, CP, STAGED>(g, s, e, in, r, ub, det, unit, anis, ua, o, lds, e0);
  hop_slot<SP, LK, R, 1, true, (3 % PK) == 0, CP, STAGED>(g, s, e, in, r, ub, det, unit, anis, ua, o, lds, e0);
  hop_slot<SP, LK, R, 1, false, (4 % PK) == 0, CP, STAGED>(g, s, e, in, r, ub, det, unit, anis, ua, o, lds, e0);
  hop_slot<SP, LK, R, 2, true, (5 % PK) == 0, CP, STAGED>(g, s, e, in, r, ub, det, unit, anis, ua, o, lds, e0);
  hop_slot<SP, LK, R, 2, false, (6 % PK) == 0, CP, STAGED>(g, s, e, in, r, ub, det, unit, anis, ua, o, lds, e0);
  hop_slot<SP, LK, R, 3, true, (7 % PK) == 0, CP, STAGED>(g, s, e, in, r, ub, det, unit, anis, ua, o, lds, e0);
  hop_slot<SP, LK, R, 3, false, true, CP, STAGED>(g, s, e, in, r, ub, det, unit, anis, ua, o, lds, e0);
}

template <int SP>
using RealOf = typename std::conditional<SP == SP_F64, double, float>::type;

// Twisted clover block (MODE 0: z + clover term, 1: inverse) of each chirality
// applied in place to the twelve components v of site e (the epilogue's block stage);
// the blocks are stored in the spinor precision SP
template <int BMODE, int SP, class R>
__device__ __forceinline__ void clover_site(const HopEpi& epi, const Geo& g, uint32_t e, cx<R> v[12])
{
  constexpr int EB = SP == SP_F64 ? 16 : (SP == SP_F32 ? 8 : 4);
  const void* B = epi.blk.data;
#pragma unroll
  for (int h = 0; h < 2; h++) {
    cx<R> w[6];
    if (epi.blk_dag) clover_half<BMODE, 1, R, EB>(B, g.stride, e, h, epi.blk_kappa, epi.blk_mu, v + 6 * h, w);
    else clover_half<BMODE, 0, R, EB>(B, g.stride, e, h, epi.blk_kappa, epi.blk_mu, v + 6 * h, w);
#pragma unroll
    for (int q = 0; q < 6; q++) v[6 * h + q] = w[q];
  }
}

// Site-local epilogue of one right-hand side r at output site e (shared by the
// one-RHS and the register-blocked kernels, so both give the same bits):
//   out_h = c1_h hop + c2_h aux + c3_h aux2, then the mode's tail; returns the
// site's contribution to the reduced norm (modes 1-3).  CLV 1: the inverse clover
// blocks act on c1 hop; CLV 2: the clover blocks act on aux (the twisted clover K).
template <int SP, int MODE, int XP, class R, int CLV = 0, int CP = kNT>
__device__ __forceinline__ double hop_epilogue(const Geo& g, const HopEpi& epi, const SpinorView& out, uint32_t e,
                                               int r, CgState* st, cx<R> o[12])
{
  using RX = RealOf<XP>;
  double nrm = 0;
  double cf[12];
  if (epi.coef) {
#pragma unroll
    for (int k = 0; k < 12; k++) cf[k] = sload(epi.coef + 12 * r + k);
  } else {
#pragma unroll
    for (int k = 0; k < 4; k++) {
      cf[k] = (&epi.c1[0][0])[k];
      cf[4 + k] = (&epi.c2[0][0])[k];
      cf[8 + k] = (&epi.c3[0][0])[k];
    }
  }
  const cx<R> c1u = mk<R>((R)cf[0], (R)cf[1]), c1l = mk<R>((R)cf[2], (R)cf[3]);
#pragma unroll
  for (int k = 0; k < 12; k++) o[k] = (k < 6 ? c1u : c1l) * o[k];
  if constexpr (CLV == 1) clover_site<1, SP, R>(epi, g, e, o);
  if (epi.aux.data) {
    cx<R> a[12];
    SpAcc<SP, R, 12, CP>::load(epi.aux, g.stride, e, a, r);
    if constexpr (CLV == 2) clover_site<0, SP, R>(epi, g, e, a);
    const cx<R> cu = mk<R>((R)cf[4], (R)cf[5]), cl = mk<R>((R)cf[6], (R)cf[7]);
#pragma unroll
    for (int k = 0; k < 12; k++) fma_to(o[k], k < 6 ? cu : cl, a[k]);
  }
  if (epi.aux2.data) {
    cx<R> a[12];
    SpAcc<SP, R, 12, CP>::load(epi.aux2, g.stride, e, a, r);
    const cx<R> cu = mk<R>((R)cf[8], (R)cf[9]), cl = mk<R>((R)cf[10], (R)cf[11]);
#pragma unroll
    for (int k = 0; k < 12; k++) fma_to(o[k], k < 6 ? cu : cl, a[k]);
  }
  if constexpr (MODE == 0) {
    SpAcc<SP, R, 12, CP>::store(out, g.stride, e, o, r);
  } else if constexpr (MODE == 1) {
    if (epi.write) SpAcc<SP, R, 12, CP>::store(out, g.stride, e, o, r);
#pragma unroll
    for (int k = 0; k < 12; k++) nrm += (double)o[k].re * (double)o[k].re + (double)o[k].im * (double)o[k].im;
  } else if constexpr (MODE == 2) {
    // CG tail: s = o; x += alpha p (when x is given) ; r -= alpha s ; |r|^2
    const RX alpha = (RX)sload(&st->alpha);
    if (epi.x.data) {
      cx<RX> x[12];
      cx<R> p[12];
      SpAcc<XP, RX, 12, CP>::load(epi.x, g.stride, e, x, r);
      SpAcc<SP, R, 12, CP>::load(epi.p, g.stride, e, p, r);
#pragma unroll
      for (int k = 0; k < 12; k++) {
        x[k].re = fma(alpha, (RX)p[k].re, x[k].re);
        x[k].im = fma(alpha, (RX)p[k].im, x[k].im);
      }
      SpAcc<XP, RX, 12, CP>::store(epi.x, g.stride, e, x, r);
    }
    cx<RX> rv[12];
    SpAcc<XP, RX, 12, CP>::load(epi.r, g.stride, e, rv, r);
#pragma unroll
    for (int k = 0; k < 12; k++) {
      rv[k].re = fma(-alpha, (RX)o[k].re, rv[k].re);
      rv[k].im = fma(-alpha, (RX)o[k].im, rv[k].im);
      nrm += (double)rv[k].re * (double)rv[k].re + (double)rv[k].im * (double)rv[k].im;
    }
    SpAcc<XP, RX, 12, CP>::store(epi.r, g.stride, e, rv, r);
  } else {
    // residual tail: r64 = o ; rs = sloppy(o) ; |o|^2
    SpAcc<SP, R, 12, CP>::store(epi.r, g.stride, e, o, r);
    if (epi.rs.data) {
      cx<RX> q[12];
#pragma unroll
      for (int k = 0; k < 12; k++) q[k] = mk<RX>((RX)o[k].re, (RX)o[k].im);
      SpAcc<XP, RX, 12, CP>::store(epi.rs, g.stride, e, q, r);
    }
#pragma unroll
    for (int k = 0; k < 12; k++) nrm += (double)o[k].re * (double)o[k].re + (double)o[k].im * (double)o[k].im;
  }
  return nrm;
}

// Whether the launch skips a right-hand side.  done and reliable are constant over the
// launch: a finalisation that rides in it (fold_finalise, mode 0) leaves its own to `stop`,
// which the CG tail right after it (mode 2) reads as well.
template <int MODE>
__device__ __forceinline__ bool rhs_idle(const CgState* st, int pred)
{
  const int reliable = sload(&st->reliable);
  const int done = sload(&st->done) | (MODE == 2 ? sload(&st->stop) : 0);
  return done || (pred == 1 && !reliable) || (pred == 2 && reliable);
}

// The workgroup past the last block finalises the previous launch's reduction (one
// right-hand side); vl: 1024 doubles of LDS.  It writes nothing that the hop reads: the
// wavefronts of a workgroup each read done and reliable, and must agree before a barrier.
// Returns true in that workgroup.
__device__ __forceinline__ bool fold_finalise(const HopEpi& epi, const double* partial, int64_t nchunks, double* vl)
{
  if (epi.fold_fin == FIN_NONE || xcd_block() != (int64_t)gridDim.x - 1) return false;
  CgState* fs = epi.st;
  if (!(fs->done || (epi.fold_pred == 1 && !fs->reliable) || (epi.fold_pred == 2 && fs->reliable))) {
    const double tot = block_sum_partials_256(partial, nchunks, vl);
    if (threadIdx.x == 0) finalize<true>(fs, epi.fold_fin, tot);
  }
  return true;
}

// workgroups of at most 256 threads; FP64 builds get the full 256-VGPR budget
// (one wavefront per SIMD per workgroup), the sloppy builds two workgroups per CU.
// FP16 pins the accumulators after every slot: the registers it saves put all of a
// middle lattice's wavefronts on the SIMDs at once.  FP16 links at 24^3x48 26.5 -> 24.1 us
// and 20^3x40 14.4 -> 13.6, FP32 links 16.3 -> 15.1 (solves 11.5 -> 11.2, 6.57 -> 6.33,
// 7.00 -> 6.86 ms), 16^3x32 equal; pins for FP32 are equal, four slots stay.
template <int SP, int LK, int MODE, int XP, int CLV = 0, int CP = kNT>
__global__ void __launch_bounds__(256, (SP != SP_F64 ? 2 : 1)) k_tm_hop(Geo g, int op, SpinorView out, SpinorView in, LinkView U, double anis_d,
                                               int use_anis, HopEpi epi, Shape S, int64_t nchunks,
                                               double* partial)
{
  using R = RealOf<SP>;
  if constexpr (MODE == 0) {
    __shared__ double vl[1024];
    if (fold_finalise(epi, partial, nchunks, vl)) return;
  }
  const Map m = map_thread(S, g.Vh);
  CgState* st = epi.st ? epi.st + m.r : nullptr;
  const bool skip = st && rhs_idle<MODE>(st, epi.pred_reliable);
  // a launch whose every right-hand side is idle does nothing (uniform over the grid)
  if (epi.st && S.NR == 1 && skip) return;
  double nrm = 0;
  if (m.active && !skip) {
    const uint32_t e = m.e;
    const int r = m.r;
    const Site s = site_of(g, op, e);
    const void* ub = U.data[op];
    const double* det = &U.det[op][0][0];
    const unsigned unit = U.unit;
    const R anis = (R)anis_d;
    const bool ua = use_anis != 0;
    cx<R> o[12];
#pragma unroll
    for (int k = 0; k < 12; k++) o[k] = mk<R>(0, 0);
    hop_site<SP, LK, R, SP == SP_F16 ? 1 : 4, CP, false>(g, s, e, in, r, ub, det, unit, anis, ua, o);
    nrm = hop_epilogue<SP, MODE, XP, R, CLV, CP>(g, epi, out, e, r, st, o);
  }
  if constexpr (MODE != 0) store_partial(nrm, partial, nchunks, m.r, m.chunk);
}

// The accumulators are pinned after every slot for FP16 (76-87 registers instead of 128,
// five or six wavefronts per SIMD beside the 13 KB of LDS: 32^3x64 hop 88 -> 85 us, FP16
// links 74 -> 61), after every two for FP64 with 12-real links (FP16 solve at 32^3x64
// 36.05 -> 35.73 ms), after every four otherwise (FP32 139 -> 132 us).
// One right-hand side, neighbours staged in LDS (Stage): the workgroup's four
// wavefronts cover 256 consecutive output sites (Shape W = 4, NRB = 1).
// The FP64 write-only hop is held to two wavefronts per SIMD: with 12-real links its
// registers would allow a third, which takes it from 240 to 243 us at 32^3x64.
template <int SP, int LK, int MODE, int XP, int CLV = 0, int CP = kNT>
__global__ void __attribute__((amdgpu_flat_work_group_size(1, 256),
                               amdgpu_waves_per_eu(SP != SP_F64 ? 2 : 1, SP == SP_F64 && MODE == 0 ? 2 : 8)))
k_tm_hop_lds(Geo g, int op, SpinorView out,
                                                                        SpinorView in, LinkView U, double anis_d,
                                                                        int use_anis, HopEpi epi, Shape S,
                                                                        int64_t nchunks, double* partial)
{
  using R = RealOf<SP>;
  __shared__ __attribute__((aligned(16))) char lds[Stage<SP, 12>::BYTES];
  static_assert(Stage<SP, 12>::BYTES >= 8192, "the finalisation needs 1024 doubles");
  if constexpr (MODE == 0) {
    if (fold_finalise(epi, partial, nchunks, (double*)lds)) return;
  }
  const Map m = map_thread(S, g.Vh);
  CgState* st = epi.st ? epi.st + m.r : nullptr;
  const bool skip = st && rhs_idle<MODE>(st, epi.pred_reliable);
  if (epi.st && skip) return;  // uniform: one right-hand side per launch
  const uint32_t e0 = (uint32_t)((m.chunk - (threadIdx.x >> 6)) * 64);  // first site of the workgroup
  const int t = (int)threadIdx.x;
  Stage<SP, 12>::put(lds, in, g.stride, e0 + t, e0 + t < (uint64_t)g.Vh, t, m.r);
  __syncthreads();
  double nrm = 0;
  if (m.active) {
    const uint32_t e = m.e;
    const int r = m.r;
    const Site s = site_of(g, op, e);
    const void* ub = U.data[op];
    const double* det = &U.det[op][0][0];
    const unsigned unit = U.unit;
    const R anis = (R)anis_d;
    const bool ua = use_anis != 0;
    cx<R> o[12];
#pragma unroll
    for (int k = 0; k < 12; k++) o[k] = mk<R>(0, 0);
    hop_site<SP, LK, R, SP == SP_F16 ? 1 : (LK == LK_F64_12 ? 2 : 4), CP, true>(g, s, e, in, r, ub, det, unit, anis, ua, o, lds, e0);
    nrm = hop_epilogue<SP, MODE, XP, R, CLV, CP>(g, epi, out, e, r, st, o);
  }
  if constexpr (MODE != 0) store_partial(nrm, partial, nchunks, m.r, m.chunk);
}

// Persistent form of k_tm_hop_lds for the FP64 hop: one resident workgroup per slot
// loops over 256-site blocks, so no SIMD idles between a finished workgroup and the
// dispatch of the next.  Its accumulators are pinned after every two slots (PK = 2:
// 176-195 VGPRs, two wavefronts per SIMD; with PK = 4 the loads of four slots in
// flight take 256 VGPRs + 32 AGPRs and one wavefront per SIMD).  Measured, hop
// alone: 24^3x48 102.2 us (PK = 2) against 106.1 (PK = 4), 32^3x64 276.0 against
// 276.5; PK = 1 (136-162 VGPRs, three wavefronts) 106 and 296 us.  The site
// body is the one of k_tm_hop_lds, written out in the same form (the compiler's
// FMA contraction follows the code's shape, and the kernels must agree bit for
// bit with each other and with k_tm_hop).  The
// workgroups of XCD x (b % 8 == x, the hardware's round-robin) walk one
// contiguous eighth of the blocks together, block bi, bi + nbx, ... of it, as the
// one-shot kernel's dispatch order does.  Partials stay per 64-site chunk.
template <int SP, int LK, int MODE, int XP, int CLV = 0>
__global__ void __launch_bounds__(256, 1) k_tm_hop_lds_p(Geo g, int op, SpinorView out, SpinorView in, LinkView U,
                                                         double anis_d, int use_anis, HopEpi epi, int64_t nblk,
                                                         int64_t nchunks, double* partial)
{
  using R = RealOf<SP>;
  __shared__ __attribute__((aligned(16))) char lds[Stage<SP, 12>::BYTES];
  CgState* st = epi.st;
  if (st && rhs_idle<MODE>(st, epi.pred_reliable)) return;  // uniform: one right-hand side per launch
  const uint32_t b = blockIdx.x, nb = gridDim.x;
  const uint32_t xcd = b & 7u, bi = b >> 3;
  const int64_t nbx = (int64_t)(nb >> 3) + (xcd < (nb & 7u) ? 1 : 0);  // workgroups on this XCD
  const int64_t q8 = nblk >> 3, r8 = nblk & 7;
  const int64_t lo = (int64_t)xcd * q8 + ((int64_t)xcd < r8 ? (int64_t)xcd : r8);
  const int64_t hi = lo + q8 + ((int64_t)xcd < r8 ? 1 : 0);
  const int t = (int)threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
  const void* ub = U.data[op];
  const double* det = &U.det[op][0][0];
  const unsigned unit = U.unit;
  const R anis = (R)anis_d;
  const bool ua = use_anis != 0;
  if constexpr (MODE == 0) {
    // No reduction, so no 64-site chunk to respect: the XCD's sites are walked in
    // rounds of 256 per workgroup, and the sites left after the last whole round
    // are split evenly over all of the XCD's workgroups and, inside each, over its
    // four wavefronts.  With whole blocks only, 24^3x48 (162 blocks per XCD on 64
    // workgroups) ends with a third round in which 30 of 64 workgroups idle.
    const int64_t s_lo = (int64_t)g.Vh * xcd / 8, n = (int64_t)g.Vh * (xcd + 1) / 8 - s_lo;
    const int64_t per_round = nbx * kStageSites, full = n / per_round;
    const int lane = t & 63;
    for (int64_t k = 0; k <= full; k++) {  // uniform over the workgroup
      int64_t e0, len;
      if (k < full) {
        e0 = s_lo + (k * nbx + bi) * kStageSites;
        len = kStageSites;
      } else {
        const int64_t rem = n - full * per_round, q = (rem + nbx - 1) / nbx;
        e0 = s_lo + full * per_round + (int64_t)bi * q;
        len = s_lo + n - e0 < q ? s_lo + n - e0 : q;
        if (len <= 0) break;
      }
      __syncthreads();  // the previous window's LDS reads are done
      Stage<SP, 12>::put(lds, in, g.stride, (uint32_t)e0 + t, e0 + t < g.Vh, t, 0);
      __syncthreads();
      const int wl = (int)((len + 3) / 4);  // sites per wavefront (64 in a whole round)
      const int64_t eo = (int64_t)wave * wl + lane;
      if (lane < wl && eo < len) {
        const uint32_t e = (uint32_t)(e0 + eo);
        const Site s = site_of(g, op, e);
        cx<R> o[12];
#pragma unroll
        for (int k2 = 0; k2 < 12; k2++) o[k2] = mk<R>(0, 0);
        hop_site<SP, LK, R, 2, kNT, true>(g, s, e, in, 0, ub, det, unit, anis, ua, o, lds, (uint32_t)e0);
        hop_epilogue<SP, MODE, XP, R, CLV>(g, epi, out, e, 0, st, o);
      }
    }
    return;
  }
  for (int64_t cb = lo + bi; cb < hi; cb += nbx) {  // uniform over the workgroup
    const uint32_t e0 = (uint32_t)(cb * kStageSites);
    __syncthreads();  // the previous block's LDS reads are done
    Stage<SP, 12>::put(lds, in, g.stride, e0 + t, e0 + t < (uint64_t)g.Vh, t, 0);
    __syncthreads();
    const uint32_t e = e0 + (uint32_t)t;
    double nrm = 0;
    if (e < (uint64_t)g.Vh) {
      const Site s = site_of(g, op, e);
      cx<R> o[12];
#pragma unroll
      for (int k = 0; k < 12; k++) o[k] = mk<R>(0, 0);
      hop_site<SP, LK, R, 2, kNT, true>(g, s, e, in, 0, ub, det, unit, anis, ua, o, lds, e0);
      nrm = hop_epilogue<SP, MODE, XP, R, CLV>(g, epi, out, e, 0, st, o);
    }
    if constexpr (MODE != 0) store_partial(nrm, partial, nchunks, 0, cb * 4 + wave);
  }
}

// resident workgroups per CU of the persistent kernel (queried once per instance)
template <int SP, int LK, int MODE, int XP, int CLV>
static int persist_per_cu()
{
  static const int occ = [] {
    int o = 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&o, (const void*)k_tm_hop_lds_p<SP, LK, MODE, XP, CLV>, 256, 0) !=
            hipSuccess || o < 1)
      o = 0;
    return o;
  }();
  return occ;
}

// ---------------------------------------------------------------- directions split over wavefronts
// FP64, one right-hand side: the four wavefronts of a workgroup take the four directions
// (two slots each) of the same 64 sites, exchange their partial sums through LDS and
// finish one spin each: wavefront w sums the four directions of spin w in the order
// t, x, y, z and runs the epilogue on its three components.  A small lattice is bound by
// the latency of one thread's chain (eight slots of loads and 1320 flops: 10 us on 8^4,
// of which 3 us are an empty launch's); four times the wavefronts with a quarter of the
// chain take it to 4.6 us (K K^+ at 12x6x10x14 66 -> 34 us, the FP64 solve at 8^3x16 4.74
// -> 2.76 ms), and on middle lattices they put more loads in flight (16^3x32 5.4 TB/s of
// compulsory bytes from the memory-side cache).  130 registers, three workgroups a CU;
// held to 128 for four it spills and was slower (16^3x32 K K^+ 90 -> 96 us).
template <int LK, int MU, int CP>
__device__ __forceinline__ void split_direction(const Geo& g, const Site& s, uint32_t e, const SpinorView& in,
                                                const void* ub, const double* det, double anis, bool ua,
                                                double2 (*xch)[3][3][64], int lane, cx<double> own[3])
{
  cx<double> o[12];
#pragma unroll
  for (int k = 0; k < 12; k++) o[k] = mk(0.0, 0.0);
  hop_slot<SP_F64, LK, double, MU, true, false, CP, false>(g, s, e, in, 0, ub, det, 0u, anis, ua, o);
  hop_slot<SP_F64, LK, double, MU, false, false, CP, false>(g, s, e, in, 0, ub, det, 0u, anis, ua, o);
#pragma unroll
  for (int k = 0; k < 12; k++) {
    if (k / 3 == MU) own[k % 3] = o[k];
    else xch[k / 3][MU < k / 3 ? MU : MU - 1][k % 3][lane] = make_double2(o[k].re, o[k].im);
  }
}

// three consecutive components of an FP64 field
template <int CP>
__device__ __forceinline__ void load3(const SpinorView& v, int64_t stride, uint32_t e, int k0, cx<double> s[3])
{
  const __amdgpu_buffer_rsrc_t rs = make_rsrc((const char*)v.data + (int64_t)k0 * stride * 16, 3 * stride * 16);
#pragma unroll
  for (int c = 0; c < 3; c++) {
    const double2 d = bload_d2<CP>(rs, e * 16u, (uint32_t)(c * stride * 16));
    s[c] = mk(d.x, d.y);
  }
}
template <int CP>
__device__ __forceinline__ void store3(const SpinorView& v, int64_t stride, uint32_t e, int k0, const cx<double> s[3])
{
#pragma unroll
  for (int c = 0; c < 3; c++)
    put<nq_dv2, CP>((nq_dv2*)((char*)v.data + ((int64_t)(k0 + c) * stride + e) * 16), nq_dv2{s[c].re, s[c].im});
}

template <int LK, int MODE, int CP>
__global__ void __launch_bounds__(256, 2) k_tm_hop_split(Geo g, int op, SpinorView out, SpinorView in, LinkView U,
                                                      double anis, int use_anis, HopEpi epi, int64_t nchunks,
                                                      double* partial)
{
  __shared__ double2 xch[4][3][3][64];  // [spin][other direction][colour][site]
  __shared__ double wsum[4];
  if constexpr (MODE == 0) {
    if (fold_finalise(epi, partial, nchunks, (double*)xch)) return;
  }
  const CgState* st = epi.st;
  if (st && rhs_idle<MODE>(st, epi.pred_reliable)) return;  // uniform: one right-hand side per launch
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int64_t chunk = xcd_block();
  const bool active = chunk * 64 + lane < g.Vh;
  // lanes past the end of a partial last chunk compute the last site and drop it
  const uint32_t e = active ? (uint32_t)(chunk * 64 + lane) : (uint32_t)(g.Vh - 1);
  const Site s = site_of(g, op, e);
  const void* ub = U.data[op];
  const double* det = &U.det[op][0][0];
  const bool ua = use_anis != 0;
  cx<double> own[3];
  if (w == 0) split_direction<LK, 0, CP>(g, s, e, in, ub, det, anis, ua, xch, lane, own);
  else if (w == 1) split_direction<LK, 1, CP>(g, s, e, in, ub, det, anis, ua, xch, lane, own);
  else if (w == 2) split_direction<LK, 2, CP>(g, s, e, in, ub, det, anis, ua, xch, lane, own);
  else split_direction<LK, 3, CP>(g, s, e, in, ub, det, anis, ua, xch, lane, own);
  // the epilogue's fields of spin w, in flight over the barrier
  const int k0 = 3 * w, hh = w >> 1;
  cx<double> a1[3], a2[3], xv[3], pv[3], rv[3];
  if (epi.aux.data) load3<CP>(epi.aux, g.stride, e, k0, a1);
  if (epi.aux2.data) load3<CP>(epi.aux2, g.stride, e, k0, a2);
  if constexpr (MODE == 2) {
    if (epi.x.data) {
      load3<CP>(epi.x, g.stride, e, k0, xv);
      load3<CP>(epi.p, g.stride, e, k0, pv);
    }
    load3<CP>(epi.r, g.stride, e, k0, rv);
  }
  __syncthreads();
  cx<double> o[3];
#pragma unroll
  for (int c = 0; c < 3; c++) {
    // directions in order, this wavefront's own in its place
    cx<double> t[3];
#pragma unroll
    for (int m = 0; m < 3; m++) t[m] = mk(xch[w][m][c][lane].x, xch[w][m][c][lane].y);
    const cx<double> d0 = w == 0 ? own[c] : t[0], d1 = w == 1 ? own[c] : (w == 0 ? t[0] : t[1]),
                     d2 = w == 2 ? own[c] : (w < 2 ? t[1] : t[2]), d3 = w == 3 ? own[c] : t[2];
    o[c] = ((d0 + d1) + d2) + d3;
  }
  const cx<double> c1 = mk(epi.c1[hh][0], epi.c1[hh][1]), c2 = mk(epi.c2[hh][0], epi.c2[hh][1]),
                   c3 = mk(epi.c3[hh][0], epi.c3[hh][1]);
#pragma unroll
  for (int c = 0; c < 3; c++) {
    o[c] = c1 * o[c];
    if (epi.aux.data) fma_to(o[c], c2, a1[c]);
    if (epi.aux2.data) fma_to(o[c], c3, a2[c]);
  }
  double nrm = 0;
  if (active) {
    if constexpr (MODE == 0) {
      store3<CP>(out, g.stride, e, k0, o);
    } else if constexpr (MODE == 1) {
      if (epi.write) store3<CP>(out, g.stride, e, k0, o);
#pragma unroll
      for (int c = 0; c < 3; c++) nrm += o[c].re * o[c].re + o[c].im * o[c].im;
    } else if constexpr (MODE == 2) {
      // CG tail: x += alpha p (when x is given) ; r -= alpha s ; |r|^2
      const double alpha = sload(&st->alpha);
      if (epi.x.data) {
#pragma unroll
        for (int c = 0; c < 3; c++) {
          xv[c].re = fma(alpha, pv[c].re, xv[c].re);
          xv[c].im = fma(alpha, pv[c].im, xv[c].im);
        }
        store3<CP>(epi.x, g.stride, e, k0, xv);
      }
#pragma unroll
      for (int c = 0; c < 3; c++) {
        rv[c].re = fma(-alpha, o[c].re, rv[c].re);
        rv[c].im = fma(-alpha, o[c].im, rv[c].im);
        nrm += rv[c].re * rv[c].re + rv[c].im * rv[c].im;
      }
      store3<CP>(epi.r, g.stride, e, k0, rv);
    } else {
      // residual tail: r64 = o ; |o|^2
      store3<CP>(epi.r, g.stride, e, k0, o);
#pragma unroll
      for (int c = 0; c < 3; c++) nrm += o[c].re * o[c].re + o[c].im * o[c].im;
    }
  }
  if constexpr (MODE != 0) {
    nrm = wave_sum(nrm);
    if (lane == 0) wsum[w] = nrm;
    __syncthreads();
    if (threadIdx.x == 0) partial[chunk] = (wsum[0] + wsum[1]) + (wsum[2] + wsum[3]);
  }
}

// The same split for the sloppy precisions and for the clover epilogues, whose FP16 norms
// and 6x6 blocks need all components of a site in one thread: the first wavefront sums the
// four directions and runs the common epilogue.
template <int SP, int LK, class R, int MU, int CP>
__device__ __forceinline__ void split_direction_to(const Geo& g, const Site& s, uint32_t e, const SpinorView& in,
                                                   const void* ub, const double* det, unsigned unit, R anis, bool ua,
                                                   cx<R> (*xch)[12][64], int lane)
{
  cx<R> o[12];
#pragma unroll
  for (int k = 0; k < 12; k++) o[k] = mk<R>(0, 0);
  hop_slot<SP, LK, R, MU, true, false, CP, false>(g, s, e, in, 0, ub, det, unit, anis, ua, o);
  hop_slot<SP, LK, R, MU, false, false, CP, false>(g, s, e, in, 0, ub, det, unit, anis, ua, o);
#pragma unroll
  for (int k = 0; k < 12; k++) xch[MU][k][lane] = o[k];
}

template <int SP, int LK, int MODE, int XP, int CLV, int CP>
__global__ void __launch_bounds__(256, 2) k_tm_hop_split_any(Geo g, int op, SpinorView out, SpinorView in, LinkView U,
                                                             double anis_d, int use_anis, HopEpi epi, int64_t nchunks,
                                                             double* partial)
{
  using R = RealOf<SP>;
  __shared__ cx<R> xch[4][12][64];  // [direction][component][site]
  static_assert(sizeof xch >= 8192, "the finalisation needs 1024 doubles");
  if constexpr (MODE == 0) {
    if (fold_finalise(epi, partial, nchunks, (double*)xch)) return;
  }
  CgState* st = epi.st;
  if (st && rhs_idle<MODE>(st, epi.pred_reliable)) return;  // uniform: one right-hand side per launch
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int64_t chunk = xcd_block();
  const bool active = chunk * 64 + lane < g.Vh;
  // lanes past the end of a partial last chunk compute the last site and drop it
  const uint32_t e = active ? (uint32_t)(chunk * 64 + lane) : (uint32_t)(g.Vh - 1);
  const Site s = site_of(g, op, e);
  const void* ub = U.data[op];
  const double* det = &U.det[op][0][0];
  const R anis = (R)anis_d;
  const bool ua = use_anis != 0;
  if (w == 0) split_direction_to<SP, LK, R, 0, CP>(g, s, e, in, ub, det, U.unit, anis, ua, xch, lane);
  else if (w == 1) split_direction_to<SP, LK, R, 1, CP>(g, s, e, in, ub, det, U.unit, anis, ua, xch, lane);
  else if (w == 2) split_direction_to<SP, LK, R, 2, CP>(g, s, e, in, ub, det, U.unit, anis, ua, xch, lane);
  else split_direction_to<SP, LK, R, 3, CP>(g, s, e, in, ub, det, U.unit, anis, ua, xch, lane);
  __syncthreads();
  if (w != 0) return;
  double nrm = 0;
  if (active) {
    cx<R> o[12];
#pragma unroll
    for (int k = 0; k < 12; k++) o[k] = ((xch[0][k][lane] + xch[1][k][lane]) + xch[2][k][lane]) + xch[3][k][lane];
    nrm = hop_epilogue<SP, MODE, XP, R, CLV, CP>(g, epi, out, e, 0, st, o);
  }
  if constexpr (MODE != 0) store_partial(nrm, partial, nchunks, 0, chunk);
}

// ---------------------------------------------------------------- register-blocked RHS
// One slot of the hop for RB right-hand sides r0..r0+nrb-1 of the same site: the
// link is loaded once and applied to each right-hand side's projected neighbour.
template <int SP, int LK, class R, int MU, bool FWD, int RB>
__device__ __forceinline__ void hop_slot_rb(const Geo& g, const Site& s, uint32_t e, const SpinorView& in, int r0,
                                            int nrb, unsigned busy, const void* ub, const double* det, unsigned unit, R anis,
                                            bool use_anis, cx<R> o[RB][12], const char* lds = nullptr,
                                            uint32_t lds_e0 = 0)
{
  const uint32_t n = neigh_eo(g, s, MU, FWD);
  cx<R> u[9];
  constexpr int slot = 2 * MU + (FWD ? 0 : 1);
  LkAcc<LK, R, kRbLinkCP>::load(ub, g.stride, slot, e, det + 2 * slot, u, lk_eb(LK) < 16 && ((unit >> MU) & 1u));
#pragma unroll
  for (int b = 0; b < RB; b++) {
    if (b >= nrb || !((busy >> b) & 1u)) continue;  // uniform over the wavefront
    cx<R> h0[3], h1[3];
    load_projected<SP, R, MU, FWD>(g, in, r0 + b, n, lds ? lds + b * Stage<SP, 12>::BYTES : nullptr, lds_e0, h0, h1);
    cx<R> g0[3], g1[3];
    mat_vec(u, h0, g0);
    mat_vec(u, h1, g1);
    if (MU > 0 && use_anis) {
#pragma unroll
      for (int c = 0; c < 3; c++) { g0[c] = scal(g0[c], anis); g1[c] = scal(g1[c], anis); }
    }
    scatter<R, MU, FWD>(o[b], g0, g1);
#pragma unroll
    for (int k = 0; k < 12; k++) asm volatile("" : "+v"(o[b][k].re), "+v"(o[b][k].im));
  }
  asm volatile("" ::: "memory");
}

// Multi-RHS hop for the sloppy precisions: wavefront w of a workgroup takes chunk
// 4*cb + w and the RB right-hand sides of group rg (Shape: W = 4, NRB = 1, NR = NRG
// = number of RB-groups).  Link traffic and link loads per right-hand side drop by RB.
// STG: the busy right-hand sides' records of the workgroup's 256 sites are staged in LDS
// and the neighbours among those sites read from there (stage_batch).
template <int SP, int LK, int MODE, int XP, int RB, bool STG>
__global__ void __launch_bounds__(256) k_tm_hop_rb(Geo g, int op, SpinorView out, SpinorView in, LinkView U,
                                                   double anis_d, int use_anis, HopEpi epi, Shape S, int nr,
                                                   int64_t nchunks, double* partial)
{
  using R = RealOf<SP>;
  const Map m = map_thread(S, g.Vh);
  const int r0 = m.r * RB, nrb = min(RB, nr - r0);
  unsigned busy = 0;
#pragma unroll
  for (int b = 0; b < RB; b++)
    if (b < nrb && !(epi.st && rhs_idle<MODE>(epi.st + r0 + b, epi.pred_reliable))) busy |= 1u << b;
  // right-hand sides that idle here are skipped by the finalisation as well
  __shared__ __attribute__((aligned(16))) char lds[STG ? RB * Stage<SP, 12>::BYTES : 16];
  const uint32_t e0 = (uint32_t)((m.chunk - (threadIdx.x >> 6)) * 64);
  if (!busy) {  // uniform over the workgroup (one right-hand-side group)
    if constexpr (MODE != 0) {
#pragma unroll
      for (int b = 0; b < RB; b++)
        if (b < nrb) store_partial(0.0, partial, nchunks, r0 + b, m.chunk);
    }
    return;
  }
  if constexpr (STG) {
#pragma unroll
    for (int b = 0; b < RB; b++)
      if (b < nrb && ((busy >> b) & 1u))
        Stage<SP, 12>::put(lds + b * Stage<SP, 12>::BYTES, in, g.stride, e0 + threadIdx.x,
                           e0 + threadIdx.x < (uint64_t)g.Vh, (int)threadIdx.x, r0 + b);
    __syncthreads();
  }
  const char* lp = STG ? lds : nullptr;
  const uint32_t e = m.e;
  cx<R> o[RB][12];
#pragma unroll
  for (int b = 0; b < RB; b++)
#pragma unroll
    for (int k = 0; k < 12; k++) o[b][k] = mk<R>(0, 0);
  // sites past the end (a partial last chunk) compute nothing but take part in the
  // wavefront reductions with zero
  if (m.active) {
    const Site s = site_of(g, op, e);
    const void* ub = U.data[op];
    const double* det = &U.det[op][0][0];
    const unsigned unit = U.unit;
    const R anis = (R)anis_d;
    const bool ua = use_anis != 0;
    hop_slot_rb<SP, LK, R, 0, true, RB>(g, s, e, in, r0, nrb, busy, ub, det, unit, anis, ua, o, lp, e0);
    hop_slot_rb<SP, LK, R, 0, false, RB>(g, s, e, in, r0, nrb, busy, ub, det, unit, anis, ua, o, lp, e0);
    hop_slot_rb<SP, LK, R, 1, true, RB>(g, s, e, in, r0, nrb, busy, ub, det, unit, anis, ua, o, lp, e0);
    hop_slot_rb<SP, LK, R, 1, false, RB>(g, s, e, in, r0, nrb, busy, ub, det, unit, anis, ua, o, lp, e0);
    hop_slot_rb<SP, LK, R, 2, true, RB>(g, s, e, in, r0, nrb, busy, ub, det, unit, anis, ua, o, lp, e0);
    hop_slot_rb<SP, LK, R, 2, false, RB>(g, s, e, in, r0, nrb, busy, ub, det, unit, anis, ua, o, lp, e0);
    hop_slot_rb<SP, LK, R, 3, true, RB>(g, s, e, in, r0, nrb, busy, ub, det, unit, anis, ua, o, lp, e0);
    hop_slot_rb<SP, LK, R, 3, false, RB>(g, s, e, in, r0, nrb, busy, ub, det, unit, anis, ua, o, lp, e0);
  }
#pragma unroll
  for (int b = 0; b < RB; b++) {
    if (b >= nrb) continue;
    double nrm = 0;
    if (m.active && ((busy >> b) & 1u)) nrm = hop_epilogue<SP, MODE, XP, R>(g, epi, out, e, r0 + b, epi.st ? epi.st + r0 + b : nullptr, o[b]);
    if constexpr (MODE != 0) store_partial(nrm, partial, nchunks, r0 + b, m.chunk);
  }
}

// ---------------------------------------------------------------- links in registers
// Batched FP16 hop: a wavefront loads the eight links of its 64 sites once, keeps rows 0
// and 1 in 96 registers and row 2 in LDS (48 KB a workgroup, each lane its own words, so
// no barrier), and loops over its right-hand sides with the records of four neighbours
// in flight, into the next right-hand side.  The register-blocked kernel rebuilt the
// links and re-read them from L2 for every one or two right-hand sides; it ran at two
// thirds of the VALU and with every slot waiting for its own loads.  Per right-hand side
// and site this leaves 120 VALU instructions a slot (12 mixed adds, 12 scalings, 72
// multiply-adds, 24 adds) of the 2159 a site took, at 224-247 registers and two wavefronts
// per SIMD.  What bounds it now is the L1's rate of misses (32^3x64: TD busy 99 %, 16 B a
// cycle and CU from L2, 2.6 times the compulsory bytes).  Twelve right-hand sides: 24^3x48 235 -> 187 us (2.9 TB/s of compulsory
// bytes), 32^3x64 692 -> 546, 16^3x32 48.5 -> 34.5; the z-tiled site order then takes
// them to 177, 517 and 35.6.  Loading all stored elements before the first rebuild and
// keeping the loop's loads unconditional matters: a load behind a branch makes every
// later wait drain the queue (616 -> 546 us).
// Slot K = 2 mu + (backward) of one FP16 neighbour applied to the accumulators.
template <int K, bool ANIS>
__device__ __forceinline__ void rl_slot(const RawF16& w, const cx<float> u6[6], const float2* row2, float anis,
                                        cx<float> o[12])
{
  cx<float> u[9];
#pragma unroll
  for (int k = 0; k < 6; k++) u[k] = u6[k];
#pragma unroll
  for (int j = 0; j < 3; j++) {
    const float2 f = row2[(3 * K + j) * 256];
    u[6 + j] = mk<float>(f.x, f.y);
  }
  constexpr int MU = K / 2;
  constexpr bool FWD = (K & 1) == 0;
  cx<float> h0[3], h1[3], g0[3], g1[3];
  project_f16<MU, FWD>(w, w.norm, h0, h1);
  mat_vec(u, h0, g0);
  mat_vec(u, h1, g1);
  // on the products, as hop_slot_rb has it: folded into the norm it rounds differently
  if constexpr (MU > 0 && ANIS) {
#pragma unroll
    for (int c = 0; c < 3; c++) { g0[c] = scal(g0[c], anis); g1[c] = scal(g1[c], anis); }
  }
  scatter<float, MU, FWD>(o, g0, g1);
  // materialise the accumulators and keep the next loads behind this slot
#pragma unroll
  for (int k = 0; k < 12; k++) asm volatile("" : "+v"(o[k].re), "+v"(o[k].im));
  asm volatile("" ::: "memory");
}

// ANIS: with an anisotropy factor (a branch on it in the loop costs every slot: twelve
// right-hand sides at 16^3x32, solve 21.2 -> 21.4 ms)
template <int LK, int MODE, int XP, int CP, bool ANIS>
__global__ void __launch_bounds__(256, 2) k_tm_hop_rl(Geo g, int op, SpinorView out, SpinorView in, LinkView U,
                                                      double anis_d, HopEpi epi, Shape S, int nr, int rpw,
                                                      int64_t nchunks, double* partial)
{
  const Map m = map_thread(S, g.Vh);
  const int r0 = m.r * rpw, r1 = min(r0 + rpw, nr);
  unsigned busy = 0;
  for (int r = r0; r < r1; r++) {
    if (epi.st && rhs_idle<MODE>(epi.st + r, epi.pred_reliable)) {
      if constexpr (MODE != 0) store_partial(0.0, partial, nchunks, r, m.chunk);
    } else {
      busy |= 1u << r;
    }
  }
  busy = __builtin_amdgcn_readfirstlane(busy);
  if (!busy) return;
  // lanes past the end of a partial last chunk compute the last site and drop it
  const uint32_t e = m.active ? m.e : (uint32_t)(g.Vh - 1);
  const Site s = site_of(g, op, e);
  uint32_t n[8];
#pragma unroll
  for (int k = 0; k < 8; k++) n[k] = neigh_eo(g, s, k / 2, (k & 1) == 0);
  __shared__ float2 lrow2[24 * 256];
  float2* row2 = lrow2 + threadIdx.x;
  using Lk = LkAcc<LK, float, CP>;
  cx<float> u[8][6];
#pragma unroll
  for (int k = 0; k < 8; k++) Lk::load_stored(U.data[op], g.stride, k, e, u[k]);
  const float anis = (float)anis_d;
  constexpr int D = 4;  // neighbours in flight
  RawF16 w[D];
  int r = __builtin_ctz(busy);
#pragma unroll
  for (int k = 0; k < D; k++) w[k].load(in, g.stride, n[k], r);
#pragma unroll
  for (int k = 0; k < 8; k++) {
    cx<float> v[9];
#pragma unroll
    for (int c = 0; c < 6; c++) v[c] = u[k][c];
    Lk::complete(&U.det[op][k][0], v, (U.unit >> (k / 2)) & 1u);
#pragma unroll
    for (int c = 0; c < 6; c++) u[k][c] = v[c];
#pragma unroll
    for (int j = 0; j < 3; j++) row2[(3 * k + j) * 256] = make_float2(v[6 + j].re, v[6 + j].im);
  }
  for (;;) {
    busy &= busy - 1;
    const int rn = busy ? __builtin_ctz(busy) : r;
    cx<float> o[12];
#pragma unroll
    for (int k = 0; k < 12; k++) o[k] = mk<float>(0, 0);
#define NQ_RL_SLOT(K)                                                              \
  rl_slot<K, ANIS>(w[K % D], u[K], row2, anis, o);                 \
  if (K + D < 8) w[K % D].load(in, g.stride, n[(K + D) % 8], r);                   \
  else w[K % D].load(in, g.stride, n[(K + D) % 8], rn);
    NQ_RL_SLOT(0) NQ_RL_SLOT(1) NQ_RL_SLOT(2) NQ_RL_SLOT(3)
    NQ_RL_SLOT(4) NQ_RL_SLOT(5) NQ_RL_SLOT(6) NQ_RL_SLOT(7)
#undef NQ_RL_SLOT
    double nrm = 0;
    if (m.active)
      nrm = hop_epilogue<SP_F16, MODE, XP, float, 0, CP>(g, epi, out, e, r, epi.st ? epi.st + r : nullptr, o);
    if constexpr (MODE != 0) store_partial(nrm, partial, nchunks, r, m.chunk);
    if (!busy) return;
    r = rn;
  }
}

// launch of the register-blocked kernel with RB right-hand sides per wavefront
// (RB = 0: the one-RHS kernel with the field-kernel shape)
template <int SP, int LK, int MODE, int XP>
static int launch_rb(nq_ctx* ctx, int RB, int op, const SpinorView& out, const SpinorView& in, const LinkView& U,
                     double anis, const HopEpi& epi, int nr)
{
  const Geo& g = ctx->geo;
  const int ua = anis != 1.0 ? 1 : 0;
  if (RB <= 0) {
    // one right-hand side per wavefront (the kernel of the unbatched operators)
    const Launch L = launch_shape(g, nr);
    NQ_HOP_LAUNCH((k_tm_hop<SP, LK, MODE, XP>), dim3((unsigned)L.blocks), dim3(L.threads), g, op,
                       out, in, U, anis, ua, epi, L.s, L.nchunks, ctx->partial);
    NQ_HIP(hipGetLastError());
    return NQ_OK;
  }
  Shape sh;
  sh.W = 4;
  sh.NRB = 1;
  sh.NRG = sh.NR = (nr + RB - 1) / RB;
  const int64_t nchunks = (g.Vh + 63) / 64;
  const dim3 grid((unsigned)((nchunks + 3) / 4 * sh.NRG)), blk(256);
#define NQ_RB(N)                                                                                                      \
  do {                                                                                                               \
    if (stage_batch(g.Vh, SP, N, nr, ctx->ncu))                                                                                  \
      NQ_HOP_LAUNCH((k_tm_hop_rb<SP, LK, MODE, XP, N, batch_stages(SP, N)>), grid, blk, g, op, out, in, U, anis, ua,  \
                    epi, sh, nr, nchunks, ctx->partial);                                                             \
    else                                                                                                             \
      NQ_HOP_LAUNCH((k_tm_hop_rb<SP, LK, MODE, XP, N, false>), grid, blk, g, op, out, in, U, anis, ua, epi, sh, nr,   \
                    nchunks, ctx->partial);                                                                          \
  } while (0)
  switch (RB) {
  case 1: NQ_RB(1); break;
  case 2: NQ_RB(2); break;
  default: NQ_RB(4); break;
  }
#undef NQ_RB
  NQ_HIP(hipGetLastError());
  return NQ_OK;
}

// launch of k_tm_hop_rl: the right-hand sides split into the fewest groups that give
// every CU its two resident workgroups (16^3x32, 12 right-hand sides: one group 42.5 us,
// two 34.5, three 36.5; 24^3x48: one group 193 us, two 198, three 205).
template <int SP, int LK, int MODE, int XP>
static int launch_rl(nq_ctx* ctx, int op, const SpinorView& out, const SpinorView& in, const LinkView& U, double anis,
                     const HopEpi& epi, int nr)
{
  if constexpr (SP == SP_F16) {
    const Geo& g = ctx->geo;
    const int64_t nchunks = (g.Vh + 63) / 64, nblk = (nchunks + 3) / 4;
    const int64_t want = std::min<int64_t>(nr, std::max<int64_t>(1, (2 * ctx->ncu + nblk - 1) / nblk));
    const int rpw = (int)((nr + want - 1) / want);
    Shape sh;
    sh.W = 4;
    sh.NRB = 1;
    sh.NRG = sh.NR = (nr + rpw - 1) / rpw;
    const dim3 grid((unsigned)(nblk * sh.NRG)), blk(256);
    const bool keep = links_stay(g.Vh, SP, LK, nr, false);
#define NQ_RL(CP, ANIS)                                                                                             \
  NQ_HOP_LAUNCH((k_tm_hop_rl<LK, MODE, XP, CP, ANIS>), grid, blk, g, op, out, in, U, anis, epi, sh, nr, rpw, nchunks, \
                ctx->partial)
    if (anis != 1.0) {
      if (keep) NQ_RL(0, true);
      else NQ_RL(kNT, true);
    } else {
      if (keep) NQ_RL(0, false);
      else NQ_RL(kNT, false);
    }
#undef NQ_RL
    NQ_HIP(hipGetLastError());
    return NQ_OK;
  } else {
    (void)ctx; (void)op; (void)out; (void)in; (void)U; (void)anis; (void)epi; (void)nr;
    return fail(NQ_EINVAL, "tm hop: links in registers need FP16 spinors");
  }
}

// Autotuner of the right-hand sides per wavefront of the batched sloppy hop: on the
// first batched launch of a (precision, batch size) it times the write-only kernel
// (no solver state, output into a scratch buffer) with RB = 1, 2 and 4 right-hand
// sides per wavefront on the caller's input and links, and keeps the fastest for
// every mode of that precision and batch size.  FP16 has k_tm_hop_rl as a further
// candidate (kTunedRl), which wins from three or four right-hand sides up and on small
// lattices: 24^3x48, one right-hand side 31.7 us register-blocked / 33.7, two 44.0 / 46.2,
// three 58.7 / 57.8, four 71 / 68, twelve 216 / 177; 32^3x64 100 / 116, 150 / 157, 208 /
// 190, -, 682 / 517; 16^3x32 12.6 / 10.1, 13.5 / 11.6, 14.9 / 15.3, 17.5 / 18.7, 42 / 36.
// It also loses where its 512 resident workgroups are filled a little more than once
// (633 blocks, three right-hand sides).  All candidates build the same per-RHS code
// (one unrolled copy per right-hand side), so the choice never changes a result; the
// one-RHS kernel (RB = 0 in launch_rb) is not a candidate: its FP16 code schedules
// the same arithmetic differently and does not give the same bits.  NQ_TUNE=0 or an
// open graph capture use RB = 2, NQ_TUNE=r k_tm_hop_rl.
constexpr int kTunedRl = 16;

template <int SP, int LK, int MODE, int XP>
static int launch_tuned(nq_ctx* ctx, int choice, int op, const SpinorView& out, const SpinorView& in,
                        const LinkView& U, double anis, const HopEpi& epi, int nr)
{
  if (choice == kTunedRl) return launch_rl<SP, LK, MODE, XP>(ctx, op, out, in, U, anis, epi, nr);
  return launch_rb<SP, LK, MODE, XP>(ctx, choice, op, out, in, U, anis, epi, nr);
}

template <int SP, int LK, int XP>
static int tuned_rb(nq_ctx* ctx, int op, const SpinorView& in, const LinkView& U, double anis, const HopEpi& epi,
                    int nr, int* rb)
{
  const std::string key = "tm_hop_rb/" + std::to_string(SP) + "/" + std::to_string(LK) + "/" + std::to_string(nr);
  auto it = ctx->tuned.find(key);
  if (it != ctx->tuned.end()) {
    *rb = it->second;
    return NQ_OK;
  }
  const char* env = getenv("NQ_TUNE");
  if (ctx->capturing || (env && env[0] == '0')) {
    *rb = 2;
    return NQ_OK;
  }
  if (SP == SP_F16 && env && env[0] == 'r') {
    *rb = kTunedRl;
    return NQ_OK;
  }
  SpinorView scratch;
  NQ_TRY(alloc_spinor_nr(ctx, "tune.out" + std::to_string(SP), SP, 12, nr, &scratch));
  HopEpi e0;
  e0.nrhs = nr;
  e0.batched = 1;
  e0.coef = epi.coef;
  const bool prof = ctx->profiling;
  ctx->profiling = false;
  hipEvent_t a, b;
  NQ_HIP(hipEventCreate(&a));
  NQ_HIP(hipEventCreate(&b));
  float best = 1e30f;
  int best_rb = 2;
  for (int cand : {1, 2, 4, kTunedRl}) {
    if (cand == kTunedRl ? SP != SP_F16 : cand > nr) continue;
    NQ_TRY((launch_tuned<SP, LK, 0, XP>(ctx, cand, op, scratch, in, U, anis, e0, nr)));  // warm-up
    NQ_HIP(hipEventRecord(a, ctx->stream));
    for (int i = 0; i < 3; i++) NQ_TRY((launch_tuned<SP, LK, 0, XP>(ctx, cand, op, scratch, in, U, anis, e0, nr)));
    NQ_HIP(hipEventRecord(b, ctx->stream));
    NQ_HIP(hipEventSynchronize(b));
    float ms = 0;
    NQ_HIP(hipEventElapsedTime(&ms, a, b));
    if (ms < best * 0.98f) {  // prefer the smaller block unless clearly slower
      best = ms;
      best_rb = cand;
    }
  }
  (void)hipEventDestroy(a);
  (void)hipEventDestroy(b);
  ctx->profiling = prof;
  ctx->tuned[key] = best_rb;
  *rb = best_rb;
  return NQ_OK;
}

// Launches the persistent staged hop and returns true when it applies: FP64
// with 18-real links and a lattice that fills the resident slots at least twice
// (measured 2.8 % faster at 32^3x64 than the one-shot kernel).  The 12-real FP64 hop runs two wavefronts
// per SIMD in the one-shot kernel and measured slower in the persistent one.
template <int SP, int LK, int MODE, int XP, int CLV>
static bool launch_persistent(nq_ctx* ctx, int op, const SpinorView& out, const SpinorView& in, const LinkView& U,
                              double anis, const HopEpi& epi, const Launch& L)
{
  if constexpr (SP == SP_F64 && LK == LK_F64_18) {
    const char* penv = getenv("NQ_PERSIST");
    if (penv && penv[0] == '0') return false;
    const int64_t nblk = (L.nchunks + 3) / 4, slots = (int64_t)ctx->ncu * persist_per_cu<SP, LK, MODE, XP, CLV>();
    if (slots < 1 || nblk < 2 * slots) return false;
    NQ_HOP_LAUNCH((k_tm_hop_lds_p<SP, LK, MODE, XP, CLV>), dim3((unsigned)slots), dim3(256),
                       ctx->geo, op, out, in, U, anis, anis != 1.0 ? 1 : 0, epi, nblk, L.nchunks, ctx->partial + epi.part0);
    return true;
  } else {
    (void)ctx; (void)op; (void)out; (void)in; (void)U; (void)anis; (void)epi; (void)L;
    return false;
  }
}

template <int SP, int LK, int MODE, int XP, int CLV = 0>
static int go(nq_ctx* ctx, int op, const SpinorView& out, const SpinorView& in, const LinkView& U, double anis,
              const HopEpi& epi, const char* name)
{
  const Geo& g = ctx->geo;
  const int nr = epi.nrhs;
  if (nr < 1 || nr > 16) return fail(NQ_EINVAL, "tm hop: right-hand sides per launch must be 1..16");
  const Launch L = launch_shape(g, nr);
  if (epi.part0 != 0 && (nr != 1 || epi.batched || epi.fin != FIN_PARTIAL))
    return fail(NQ_EINVAL, "tm hop: a partial offset needs one right-hand side and FIN_PARTIAL");
  if (epi.part0 < 0 || epi.part0 + L.nchunks * nr > ctx->max_partials) return fail(NQ_EINVAL, "tm hop: reduction scratch too small");
  if constexpr (MODE != 3 && CLV == 0) {
    if (epi.batched || nr > 1) {
      // register-blocked right-hand sides (always for batched solves, so that a
      // right-hand side runs the same code alone and in a batch); RB right-hand
      // sides per wavefront, chosen by the autotuner for this precision and batch.
      // FP64 too: the reliable updates of a batch share each link load (measured
      // 953 -> 879 us for 12 sources, the batched FP64 solve 95 -> 85 ms per source)
      int RB = 0;
      NQ_TRY((tuned_rb<SP, LK, XP>(ctx, op, in, U, anis, epi, nr, &RB)));
      prof_begin_ext(ctx, name, tm_hop_bytes(SP, LK, epi) * (double)g.Vh, &ctx->hop_ev[0], &ctx->hop_ev[1]);
      const int rc = launch_tuned<SP, LK, MODE, XP>(ctx, RB, op, out, in, U, anis, epi, nr);
      prof_end_ext(ctx);
      NQ_TRY(rc);
      if (epi.fold_fin != FIN_NONE) NQ_TRY(launch_finalize(ctx, nr, epi.st, epi.fold_fin, epi.fold_pred));
      if (MODE != 0 && epi.fin != FIN_PARTIAL) NQ_TRY(launch_finalize(ctx, nr, epi.st, epi.fin, epi.pred_reliable));
      return NQ_OK;
    }
  }
  prof_begin_ext(ctx, name, tm_hop_bytes(SP, LK, epi) * (double)g.Vh, &ctx->hop_ev[0], &ctx->hop_ev[1]);
  bool fold_here = false;
  const char* lenv = getenv("NQ_LDS");
  // one extra workgroup carries the finalisation of the previous reduction when the
  // workgroups have 256 threads; the kernel sees fold_fin only then
  HopEpi ke = epi;
  fold_here = MODE == 0 && epi.fold_fin != FIN_NONE && nr == 1 && epi.st && L.threads == 256;
  if (!fold_here) ke.fold_fin = FIN_NONE;
  const dim3 grid((unsigned)(L.blocks + (fold_here ? 1 : 0))), blk(L.threads);
  const int ua = anis != 1.0 ? 1 : 0;
  const HopRoute route = hop_route(g.Vh, SP, LK, XP, CLV != 0, nr, epi.coef != nullptr, !(lenv && lenv[0] == '0'));
  const bool keep = route.keep, lds_ok = route.kernel == HOP_LDS;
  if (route.kernel == HOP_SPLIT) {
    // the specialised FP64 kernel has no precision conversion and no clover blocks
    constexpr bool plain64 = SP == SP_F64 && XP == SP_F64 && CLV == 0;
    HopEpi ks = epi;
    fold_here = MODE == 0 && epi.fold_fin != FIN_NONE && epi.st;
    if (!fold_here) ks.fold_fin = FIN_NONE;
    const dim3 sg((unsigned)(L.nchunks + (fold_here ? 1 : 0)));
    double* part = ctx->partial + epi.part0;
    if constexpr (plain64) {
      if (keep)
        NQ_HOP_LAUNCH((k_tm_hop_split<LK, MODE, 0>), sg, dim3(256), g, op, out, in, U, anis, ua, ks, L.nchunks, part);
      else
        NQ_HOP_LAUNCH((k_tm_hop_split<LK, MODE, kNT>), sg, dim3(256), g, op, out, in, U, anis, ua, ks, L.nchunks, part);
    } else {
      // links that do not stay: only those of the FP64 residual hop, on the lattices split here
      constexpr int NK = SP == SP_F64 && MODE == 3 ? kNT : 0;
      if (keep)
        NQ_HOP_LAUNCH((k_tm_hop_split_any<SP, LK, MODE, XP, CLV, 0>), sg, dim3(256), g, op, out, in, U, anis, ua, ks,
                      L.nchunks, part);
      else
        NQ_HOP_LAUNCH((k_tm_hop_split_any<SP, LK, MODE, XP, CLV, NK>), sg, dim3(256), g, op, out, in, U, anis, ua, ks,
                      L.nchunks, part);
    }
    prof_end_ext(ctx);
    NQ_HIP(hipGetLastError());
    if (epi.fold_fin != FIN_NONE && !fold_here) NQ_TRY(launch_finalize(ctx, 1, epi.st, epi.fold_fin, epi.fold_pred));
    if (MODE != 0 && epi.fin != FIN_PARTIAL) NQ_TRY(launch_finalize(ctx, nr, epi.st, epi.fin, epi.pred_reliable));
    return NQ_OK;
  }
  // with the default policy only where hop_route can come to it
  constexpr int KL = hop_lds_keeps(SP, MODE, CLV != 0) ? 0 : kNT;
  if (lds_ok && launch_persistent<SP, LK, MODE, XP, CLV>(ctx, op, out, in, U, anis, epi, L)) {
    fold_here = false;
  } else if (lds_ok && keep) {
    NQ_HOP_LAUNCH((k_tm_hop_lds<SP, LK, MODE, XP, CLV, KL>), grid, blk, g, op, out, in, U, anis, ua, ke, L.s, L.nchunks,
                  ctx->partial + epi.part0);
  } else if (lds_ok) {
    NQ_HOP_LAUNCH((k_tm_hop_lds<SP, LK, MODE, XP, CLV, kNT>), grid, blk, g, op, out, in, U, anis, ua, ke, L.s,
                  L.nchunks, ctx->partial + epi.part0);
  } else if (keep) {
    NQ_HOP_LAUNCH((k_tm_hop<SP, LK, MODE, XP, CLV, 0>), grid, blk, g, op, out, in, U, anis, ua, ke, L.s, L.nchunks,
                  ctx->partial + epi.part0);
  } else {
    NQ_HOP_LAUNCH((k_tm_hop<SP, LK, MODE, XP, CLV, kNT>), grid, blk, g, op, out, in, U, anis, ua, ke, L.s, L.nchunks,
                  ctx->partial + epi.part0);
  }
  prof_end_ext(ctx);
  NQ_HIP(hipGetLastError());
  if (epi.fold_fin != FIN_NONE && !fold_here) NQ_TRY(launch_finalize(ctx, 1, epi.st, epi.fold_fin, epi.fold_pred));
  if (MODE != 0 && epi.fin != FIN_PARTIAL) NQ_TRY(launch_finalize(ctx, nr, epi.st, epi.fin, epi.pred_reliable));
  return NQ_OK;
}

#define NQ_MODES(SP, LK, XP, TAG)                                                            \
  switch (epi.mode) {                                                                       \
  case 0: return go<SP, LK, 0, SP>(ctx, op, out, in, U, anis, epi, "tm_hop_" TAG);            \
  case 1: return go<SP, LK, 1, SP>(ctx, op, out, in, U, anis, epi, "tm_hop_norm_" TAG);       \
  case 2: return go<SP, LK, 2, XP>(ctx, op, out, in, U, anis, epi, "tm_hop_cgtail_" TAG);     \
  default: break;                                                                           \
  }

// Twisted clover K: the first hop with the inverse blocks (blk_mode 1, mode 0 only)
// and the second with the clover blocks on aux (blk_mode 2, modes 0-2), for the
// operator precisions of the clover solves: FP64 spinors with FP64 18-real links and
// FP64 blocks; FP32 spinors with FP32 18-real links and FP32 blocks; FP16 spinors
// with FP32 or FP16 12-real links and FP16 blocks.
template <int SP, int LK, int XP>
static int clover_modes(nq_ctx* ctx, int op, const SpinorView& out, const SpinorView& in, const LinkView& U,
                        double anis, const HopEpi& epi, const char* tag)
{
  const std::string n1 = std::string("tm_hop_clinv_") + tag, n0 = std::string("tm_hop_cldee_") + tag,
                    nn = std::string("tm_hop_norm_cldee_") + tag, nt = std::string("tm_hop_cgtail_cldee_") + tag;
  if (epi.blk_mode == 1 && epi.mode == 0) return go<SP, LK, 0, SP, 1>(ctx, op, out, in, U, anis, epi, n1.c_str());
  if (epi.blk_mode == 2) {
    if (!epi.aux.data) return fail(NQ_EINVAL, "tm hop: clover blocks on aux without aux");
    switch (epi.mode) {
    case 0: return go<SP, LK, 0, SP, 2>(ctx, op, out, in, U, anis, epi, n0.c_str());
    case 1: return go<SP, LK, 1, SP, 2>(ctx, op, out, in, U, anis, epi, nn.c_str());
    case 2: return go<SP, LK, 2, XP, 2>(ctx, op, out, in, U, anis, epi, nt.c_str());
    default: break;
    }
  }
  return fail(NQ_EINVAL, "tm hop: clover epilogue %d with mode %d", epi.blk_mode, epi.mode);
}

}  // namespace nq
