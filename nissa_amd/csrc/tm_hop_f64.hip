// Twisted-mass hop, FP64 spinors and 18-real FP64 links.

#include "tm_hop_kernels.hpp"
#include "tm_hop_prec.hpp"

namespace nq {

int tm_hop_f64(NQ_TM_HOP_ARGS)
{
  if (epi.blk_mode) return clover_modes<SP_F64, LK_F64_18, SP_F64>(ctx, op, out, in, U, anis, epi, "f64");
  if (epi.mode == 2 && epi.r.prec != SP_F64) return fail(NQ_EINVAL, "FP64 CG tail needs FP64 x,r");
  NQ_MODES(SP_F64, LK_F64_18, SP_F64, "f64")
  if (epi.mode == 3) {
    if (epi.r.prec != SP_F64) return fail(NQ_EINVAL, "residual tail needs FP64 r");
    if (!epi.rs.data) return go<SP_F64, LK_F64_18, 3, SP_F64>(ctx, op, out, in, U, anis, epi, "tm_hop_res_f64");
    if (epi.rs.prec == SP_F32) return go<SP_F64, LK_F64_18, 3, SP_F32>(ctx, op, out, in, U, anis, epi, "tm_hop_res_f64_s32");
    if (epi.rs.prec == SP_F16) return go<SP_F64, LK_F64_18, 3, SP_F16>(ctx, op, out, in, U, anis, epi, "tm_hop_res_f64_s16");
  }
  return fail(NQ_EINVAL, "tm hop: unsupported precision combination (spinor %d, links %d, mode %d)", in.prec, U.prec,
              epi.mode);
}

}  // namespace nq
