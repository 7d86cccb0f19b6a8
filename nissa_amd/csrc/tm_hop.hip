// Dispatch of the twisted-mass hop (tm_hop_kernels.hpp) over the storage precisions; the
// instances of each precision are compiled in a file of their own (tm_hop_<prec>.hip).

#include "nq_device.hpp"
#include "tm_hop_prec.hpp"

namespace nq {

static double sp_site_bytes(int sp, int ncomp)
{
  switch (sp) {
  case SP_F64: return 16.0 * ncomp;
  case SP_F32: return 8.0 * ncomp;
  default: return 4.0 * ncomp + 4.0;
  }
}
static double lk_bytes(int lk)
{
  switch (lk) {
  case LK_F64_18: return 144;
  case LK_F32_18: return 72;
  case LK_F32_12: return 48;
  case LK_F64_12: return 96;
  default: return 24;
  }
}

static int xp_of(const HopEpi& epi, int sp)
{
  if (epi.mode == 2) return epi.r.prec;
  if (epi.mode == 3) return epi.rs.data ? epi.rs.prec : sp;
  return sp;
}

double tm_hop_bytes(int sp, int lk, const HopEpi& epi, int ncomp)
{
  // per output site: the 8 links once for all right-hand sides, everything else per RHS
  const double s = sp_site_bytes(sp, ncomp);
  double b = s;  // input spinor (each site read once)
  if (epi.aux.data) b += s;
  if (epi.aux2.data) b += s;
  if (epi.mode == 0 || (epi.mode == 1 && epi.write)) b += s;
  if (epi.mode == 2) {
    const double sx = sp_site_bytes(xp_of(epi, sp), ncomp);
    b += epi.x.data ? 4 * sx + s : 2 * sx;  // r (and x) read+write, p read
  }
  if (epi.mode == 3) {
    b += s;
    if (epi.rs.data) b += sp_site_bytes(epi.rs.prec, ncomp);
  }
  // clover blocks of the epilogue: 72 (inverse) or 36 complex per site in the spinor
  // precision, read once for all right-hand sides
  const double blk = epi.blk_mode ? (epi.blk_mode == 1 ? 72.0 : 36.0) * (sp == SP_F64 ? 16 : (sp == SP_F32 ? 8 : 4)) : 0.0;
  return 8 * lk_bytes(lk) + blk + b * epi.nrhs;
}

int64_t blocks_for(int64_t n) { return (n + kBlock - 1) / kBlock; }

int launch_tm_hop(nq_ctx* ctx, int op, const SpinorView& out, const SpinorView& in, const LinkView& U, double anis,
                  const HopEpi& epi)
{
  if (in.ncomp != 12) return fail(NQ_EINVAL, "tm hop needs spincolor fields");
  if (epi.mode != 0 && !epi.st) return fail(NQ_EINVAL, "reducing epilogue without state");
  const int sp = in.prec, lk = U.prec;
  if ((epi.mode == 0 || (epi.mode == 1 && epi.write)) && out.prec != sp)
    return fail(NQ_EINVAL, "tm hop: output precision differs from input");
  if (epi.aux.data && epi.aux.prec != sp) return fail(NQ_EINVAL, "tm hop: aux precision mismatch");
  if (epi.aux2.data && epi.aux2.prec != sp) return fail(NQ_EINVAL, "tm hop: aux2 precision mismatch");
  if (epi.mode == 2 && (epi.p.prec != sp || (epi.x.data && epi.x.prec != epi.r.prec)))
    return fail(NQ_EINVAL, "tm hop: CG tail precision mismatch");
  if (epi.blk_mode && (!epi.blk.data || epi.blk.prec != sp || epi.blk.ncomp != (epi.blk_mode == 1 ? 72 : 36)))
    return fail(NQ_EINVAL, "tm hop: clover blocks of the wrong kind or precision");
  if (sp == SP_F64 && lk == LK_F64_18) return tm_hop_f64(ctx, op, out, in, U, anis, epi);
  if (sp == SP_F64 && lk == LK_F64_12 && !epi.blk_mode) return tm_hop_f64_l64c(ctx, op, out, in, U, anis, epi);
  if (sp == SP_F32 && lk == LK_F32_18) return tm_hop_f32(ctx, op, out, in, U, anis, epi);
  if (sp == SP_F16 && lk == LK_F32_12) return tm_hop_f16_l32c(ctx, op, out, in, U, anis, epi);
  if (sp == SP_F16 && lk == LK_F16_12) return tm_hop_f16_l16c(ctx, op, out, in, U, anis, epi);
  if (epi.blk_mode) return fail(NQ_EINVAL, "tm hop: no clover epilogue for spinor precision %d with links %d", sp, lk);
  return fail(NQ_EINVAL, "tm hop: unsupported precision combination (spinor %d, links %d, mode %d)", sp, lk, epi.mode);
}

}  // namespace nq
