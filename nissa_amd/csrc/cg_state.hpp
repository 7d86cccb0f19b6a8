// Solver states of the CG recurrences and their updates.  Free of HIP, so that a host
// compiler builds the recurrences as the kernels run them.
#pragma once

#include <cmath>

#if defined(__HIPCC__)
#define NQ_HD __host__ __device__
#else
#define NQ_HD
#endif

namespace nq {

// Solver state living in device memory; updated by the finalisation kernel
// that follows each reducing launch.
struct CgState {
  double b2, target;
  double rr, rr_new, pAp, alpha, beta;
  double r0, delta;     // reliable-update reference |r| and threshold factor
  double true_rr;       // last FP64 residual
  double extra[6];
  double alpha_prev;    // alpha of the previous iteration (paired x updates)
  // pending: a finalisation (Fin) of rr_new that the p update has acted on (launch_cg_pupdate
  // with fin) and that the next FIN_PAP finalisation or launch_cg_commit records
  int iter, niter, done, reliable, nreliable, nan, mixed, pending;
  // done (bit 0) or reliable (bit 1) as raised by a finalisation that rides in a hop, whose
  // other workgroups read done and reliable: the CG tail and the reductions after that hop
  // idle on either, and the finalisation of |r|^2 that follows, or the p update in its
  // place, turns it into done and reliable, for every later launch.  launch_cg_commit
  // clears it.
  int stop;
  // paired x updates of the one-source mixed CG: xlag = the last p update left its
  // alpha p term to the next one; xstep = the coming p update applies both terms
  int xlag, xstep;
};

constexpr int kMaxShift = 16;

// Multi-shift CG state of one source (cgm_invert recurrences); lives in device
// memory, updated by the CGM finalisation kernels.
// Mixed precision (mixed = 1): the sloppy solutions are flushed into FP64 and the
// Krylov residual is replaced by the FP64 residual of the hardest running shift
// (kref, the smallest running shift) whenever that shift's squared residual has
// dropped by delta2 since the last such update.  reliable = 1: flagged at the end of an iteration
// whose p/ps update still runs; 2: idle until the host's update clears it.
struct CgmState {
  double b2, rr, betaa, betap, alpha, rfrf, pap, rel_ref, delta2, pad0;
  double shift[kMaxShift], target[kMaxShift], zps[kMaxShift], zas[kMaxShift], zfs[kMaxShift];
  double betas[kMaxShift], alphas[kMaxShift], res[kMaxShift];
  double betas_prev[kMaxShift];  // betas_k of the previous iteration (paired sol_k updates)
  int run[kMaxShift];
  // owe_k: the sol_k term betas_k ps_k of the last hop2 is still to be applied,
  // 1 by the host's settle kernel (the shift stopped or the source ended), 2 by
  // the update kernel (a reliable update follows)
  int owe[kMaxShift];
  int done, reliable;  // adjacent: the sloppy kernels skip a source when either is set
  int nshift, nrun, iter, niter, nan, mixed, kref, nreliable;
  // lx solves (launch_cgm_vec): the shift vectors are updated every other iteration, from
  // the pending iteration's coefficients (b1, z1, a1; ran1: shifts that ran in it; ran2:
  // in the current one).  vmode, set by the rfrf finalisation, is the next vector
  // update's work: 0 none (idle after the end), 1 p only, keeping r (this iteration stays
  // pending), 2 p and both iterations, 3 the last iteration alone (the end came on one)
  double b1[kMaxShift], z1[kMaxShift], a1[kMaxShift];
  int ran1[kMaxShift], ran2[kMaxShift];
  int lx, vlag, vmode, pad1;
  // pend: the ps_k update of the iteration just finalised is left to the next
  // iteration's hop2 kernel (set by the rfrf finalisation when the source goes on
  // without a reliable update; the update kernel then updates p only)
  // lag: the last hop2 left its sol_k terms to the next one, which applies both
  // iterations' terms in order (so sol_k is read and written every other iteration)
  int pend, lag;
};

enum Fin {
  FIN_NONE = 0,
  FIN_STORE0 = 1,     // extra[0] = total
  FIN_PAP = 2,        // pAp = total; alpha = rr/pAp
  FIN_RR = 3,         // plain CG: beta, rr, iter, done
  FIN_RR_SLOPPY = 4,  // mixed CG: decide reliable update
  FIN_RR_TRUE = 5,    // mixed CG: after FP64 recomputation
  FIN_RR_INIT = 6,    // initial residual: rr = total, r0 = sqrt
  FIN_STORE1 = 7,     // extra[1] = total
  FIN_RR_TRUE_HOLD = 8,  // as FIN_RR_TRUE, but `reliable` stays raised (batched updates)
  FIN_INIT_B2 = 9,    // start of a solve on r = b: b2 = rr = total, target *= total
  FIN_PARTIAL = 10,   // leave the per-chunk partials for a caller's own finalisation
};

// done (bit 0) and reliable (bit 1) raised by a finalisation; RIDING: one that shares a
// launch with readers of both leaves them in `stop` (CgState)
template <bool RIDING>
NQ_HD inline void raise_stop(CgState* st, int bits)
{
  if (RIDING) {
    st->stop |= bits;
  } else {
    if (bits & 1) st->done = 1;
    if (bits & 2) st->reliable = 1;
  }
}

// One recurrence of the CG / mixed CG.
template <bool RIDING>
NQ_HD inline void record(CgState* st, int fin, double total)
{
  using std::isnan;
  using std::sqrt;
  switch (fin) {
  case FIN_STORE0: st->extra[0] = total; break;
  case FIN_STORE1: st->extra[1] = total; break;
  case FIN_PAP:
    st->pAp = total;
    st->alpha_prev = st->alpha;
    st->alpha = st->rr / total;
    if (!(total > 0.0) || isnan(total)) { st->nan = 1; raise_stop<RIDING>(st, 1); }
    break;
  case FIN_RR: {
    const double rr_new = total;
    st->iter += 1;
    st->beta = rr_new / st->rr;
    st->rr = rr_new;
    if (isnan(st->beta)) { st->nan = 1; raise_stop<RIDING>(st, 1); }
    if (!(rr_new >= st->target) || st->iter >= st->niter) raise_stop<RIDING>(st, 1);
    break;
  }
  case FIN_RR_SLOPPY: {
    // mixed CG: when |r| has dropped by delta since the last FP64 residual (or the
    // sloppy residual reached the target, or the iteration budget is spent) raise
    // `reliable`: the sloppy kernels then idle until the host has run the FP64
    // reliable update, whose finalisation (FIN_RR_TRUE) clears it again.
    const double rr_new = total;
    st->iter += 1;
    st->rr_new = rr_new;
    if (isnan(rr_new)) { st->nan = 1; raise_stop<RIDING>(st, 1); break; }
    if (sqrt(rr_new) < st->delta * st->r0 || rr_new < st->target || st->iter >= st->niter) {
      raise_stop<RIDING>(st, 2);
    } else {
      st->beta = rr_new / st->rr;
      st->rr = rr_new;
      // paired x updates: this p update applies two terms when the last one left its own
      st->xstep = st->xlag;
      st->xlag = !st->xlag;
    }
    break;
  }
  case FIN_RR_TRUE:
  case FIN_RR_TRUE_HOLD: {
    const double rr_true = total;
    st->nreliable += 1;
    st->true_rr = rr_true;
    st->beta = rr_true / st->rr;
    st->rr = rr_true;
    st->r0 = sqrt(rr_true);
    st->xlag = 0;  // the reliable update has taken every x term
    if (fin == FIN_RR_TRUE) st->reliable = 0;
    if (isnan(rr_true)) { st->nan = 1; st->done = 1; }
    if (rr_true < st->target || st->iter >= st->niter) st->done = 1;
    break;
  }
  case FIN_INIT_B2:
    st->b2 = total;
    st->target *= total;
    st->rr = total;
    st->r0 = sqrt(total);
    st->true_rr = total;
    if (!(total > 0.0) || isnan(total)) { st->nan = 1; st->done = 1; }
    break;
  case FIN_RR_INIT:
    st->rr = total;
    st->r0 = sqrt(total);
    st->true_rr = total;
    if (isnan(total)) { st->nan = 1; st->done = 1; }
    if (!(total >= st->target)) st->done = 1;
    break;
  default: break;
  }
}

// FIN_PAP first records a finalisation that the p update left pending; when that one
// stops the source or raises `reliable`, alpha stays.
template <bool RIDING = false>
NQ_HD inline void finalize(CgState* st, int fin, double total)
{
  if (fin == FIN_PAP && st->pending) {
    const int f = st->pending;
    st->pending = FIN_NONE;
    record<RIDING>(st, f, st->rr_new);
    if (st->stop || st->done || st->reliable) return;
  }
  record<RIDING>(st, fin, total);
}

// iterations to enqueue before the next poll, from the observed convergence rate: 2 to 64,
// or last_chunk before there is one
inline int next_chunk(double rr0, double rr, double target, int done_iters, int last_chunk)
{
  if (done_iters <= 0 || !(rr > 0) || !(rr0 > rr)) return last_chunk;
  const double rate = std::log(rr / rr0) / done_iters;  // log decrease per iteration (<0)
  const double need = std::ceil(std::log(target / rr) / rate) + 1;
  return need < 2 ? 2 : (need < 64 ? (int)need : 64);  // 64 for a target of zero
}

// the same for a multi-shift solve with relative residuals: the running shift that needs
// most (the targets are each shift's own, so that is not always the smallest shift)
inline int next_chunk_cgm(const CgmState& s, int last_chunk)
{
  int n = 0;
  for (int k = 0; k < s.nshift; k++) {
    if (!s.run[k]) continue;
    const int c = next_chunk(1.0, s.res[k], s.target[k], s.iter, last_chunk);
    n = c > n ? c : n;
  }
  return n > 0 ? n : last_chunk;
}

}  // namespace nq
