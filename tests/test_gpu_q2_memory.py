"""Scratch memory of the multi-mass CG on Q^2: r, p, t, s and two fields per mass."""
import numpy as np
import pytest
import torch

import nissa_amd as nq
from helpers import tm_conf

pytestmark = pytest.mark.gpu


def test_q2_multi_mass_scratch():
    L = (16, 32, 32, 32)
    field = int(np.prod(L)) * 192  # bytes of an FP64 spinor field
    with nq.Ctx(L) as ctx:
        g = nq.Gauge(ctx, lx=tm_conf(L, 4))
        src = ctx.field(nq.SPINCOLOR, nq.LX, nq.source_lx(L, 5))
        sol = ctx.field(nq.SPINCOLOR, nq.LX)
        nq.tm_apply_Q(ctx, g, 0.16, 0.1, sol, src)  # builds the links
        ctx.sync()
        free = torch.cuda.mem_get_info()[0]
        nq.tmQ2_cgm(ctx, g, 0.16, [0.1], 2, [1e-24], [sol], src)
        ctx.sync()
        used = free - torch.cuda.mem_get_info()[0]
        assert used < 6.5 * field, used / field
