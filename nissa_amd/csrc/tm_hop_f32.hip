// Twisted-mass hop, FP32 spinors and 18-real FP32 links.

#include "tm_hop_kernels.hpp"
#include "tm_hop_prec.hpp"

namespace nq {

int tm_hop_f32(NQ_TM_HOP_ARGS)
{
  if (epi.blk_mode) return clover_modes<SP_F32, LK_F32_18, SP_F32>(ctx, op, out, in, U, anis, epi, "f32");
  if (epi.mode == 2 && epi.r.prec != SP_F32) return fail(NQ_EINVAL, "FP32 CG tail needs FP32 x,r");
  NQ_MODES(SP_F32, LK_F32_18, SP_F32, "f32")
  return fail(NQ_EINVAL, "tm hop: unsupported precision combination (spinor %d, links %d, mode %d)", in.prec, U.prec,
              epi.mode);
}

}  // namespace nq
