// Twisted-mass hop, FP16 spinors and 12-real FP16 links.

#include "tm_hop_kernels.hpp"
#include "tm_hop_prec.hpp"

namespace nq {

int tm_hop_f16_l16c(NQ_TM_HOP_ARGS)
{
  if (epi.blk_mode) return clover_modes<SP_F16, LK_F16_12, SP_F32>(ctx, op, out, in, U, anis, epi, "f16_l16c");
  if (epi.mode == 2 && epi.r.prec != SP_F32) return fail(NQ_EINVAL, "FP16 CG tail needs FP32 x,r");
  NQ_MODES(SP_F16, LK_F16_12, SP_F32, "f16_l16c")
  return fail(NQ_EINVAL, "tm hop: unsupported precision combination (spinor %d, links %d, mode %d)", in.prec, U.prec,
              epi.mode);
}

}  // namespace nq
