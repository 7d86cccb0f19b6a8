// The twisted-mass hop of one storage precision each (tm_hop_<prec>.hip).
#pragma once

#include "nq_internal.hpp"

namespace nq {

#define NQ_TM_HOP_ARGS                                                                                      \
  nq_ctx *ctx, int op, const SpinorView &out, const SpinorView &in, const LinkView &U, double anis, const HopEpi &epi
int tm_hop_f64(NQ_TM_HOP_ARGS);       // FP64 spinors, 18-real FP64 links
int tm_hop_f64_l64c(NQ_TM_HOP_ARGS);  // FP64 spinors, 12-real FP64 links
int tm_hop_f32(NQ_TM_HOP_ARGS);       // FP32 spinors, 18-real FP32 links
int tm_hop_f16_l32c(NQ_TM_HOP_ARGS);  // FP16 spinors, 12-real FP32 links
int tm_hop_f16_l16c(NQ_TM_HOP_ARGS);  // FP16 spinors, 12-real FP16 links

}  // namespace nq
