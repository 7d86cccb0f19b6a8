"""Variants of the twisted-mass hop kernels at the sizes where their dispatch changes.

* The batched FP16 hop keeps the links of a site in registers and loops over its
  right-hand sides, in one or several groups; the tuner may take the register-blocked
  kernel instead.  A source has the same bits alone and
  in a batch whichever kernel and grouping the batch size picks, and small lattices agree
  with the oracle (1e-10, the bar of the other mixed solves at residue 1e-24).
* Links with a phase in every direction (the det of each slot enters the third row) and
  with a phase in t alone (it is left out elsewhere).
* The staggered batch: same bits however many sources a wavefront takes.
* Site orders whose z tile does not fit the extent (2 mod 4) or spans it.
"""
import numpy as np
import pytest

import nissa_amd as nq
from helpers import gauss_eo, rel_l2, st_conf
from oracle import oracle as orc

pytestmark = pytest.mark.gpu


def conf_of(L, seed, theta):
    conf = nq.gauge_random_lx(L, seed, 0.3)
    nq.gauge_phase_lx(L, conf, theta)
    return conf


# 16^3x32 splits five right-hand sides into two groups
@pytest.mark.parametrize("L,nr", [((32, 16, 16, 16), 5), ((16, 32, 32, 32), 3)])
@pytest.mark.parametrize("prec", ["f16", "f16h"])
def test_batched_f16_same_bits_alone(L, nr, prec):
    conf = conf_of(L, 51, [1.0, 0, 0, 0])
    with nq.Ctx(L) as ctx:
        g = nq.Gauge(ctx, lx=conf)
        src = [ctx.field(nq.SPINCOLOR, nq.LX, nq.source_lx(L, 60 + i)) for i in range(nr)]
        sol = [ctx.field(nq.SPINCOLOR, nq.LX) for _ in range(nr)]
        mus = [0.02 + 0.01 * i for i in range(nr)]
        res = nq.tm_solve_eoprec_multi(ctx, g, 0.16, mus, 1000, 1e-14, sol, src, prec=prec)
        assert all(r["rc"] == nq.NQ_OK and r["rel_res_sq"] < 2e-14 for r in res), res
        for i in (0, nr - 1):
            one = [ctx.field(nq.SPINCOLOR, nq.LX)]
            nq.tm_solve_eoprec_multi(ctx, g, 0.16, mus[i:i + 1], 1000, 1e-14, one, src[i:i + 1], prec=prec)
            assert np.array_equal(one[0].download(), sol[i].download()), i


# the register-blocked kernel (NQ_TUNE=0) and the one with the links in registers
# (NQ_TUNE=r), whichever the tuner would take: every epilogue of a solve, same bits
@pytest.mark.parametrize("L,nr", [((10, 4, 2, 2), 3), ((32, 16, 16, 16), 5), ((46, 16, 22, 20), 2)])
@pytest.mark.parametrize("prec", ["f16", "f16h"])
def test_batched_f16_kernels_agree(L, nr, prec, monkeypatch):
    conf = conf_of(L, 55, [1.0, 0.2, 0, 0])
    sols = []
    for tune in ("0", "r"):
        monkeypatch.setenv("NQ_TUNE", tune)
        with nq.Ctx(L) as ctx:
            g = nq.Gauge(ctx, lx=conf)
            src = [ctx.field(nq.SPINCOLOR, nq.LX, nq.source_lx(L, 90 + i)) for i in range(nr)]
            sol = [ctx.field(nq.SPINCOLOR, nq.LX) for _ in range(nr)]
            res = nq.tm_solve_eoprec_multi(ctx, g, 0.16, [0.05] * nr, 1000, 1e-14, sol, src, prec=prec)
            assert all(r["rc"] == nq.NQ_OK for r in res), res
            sols.append([f.download() for f in sol])
    for i in range(nr):
        assert np.array_equal(sols[0][i], sols[1][i]), i


# an anisotropy factor scales the products of the x, y and z links: same bits from both
# kernels, and alone as in the batch
@pytest.mark.parametrize("L,nr", [((10, 4, 2, 2), 3), ((32, 16, 16, 16), 5)])
@pytest.mark.parametrize("prec", ["f16", "f16h"])
def test_batched_f16_kernels_agree_anisotropic(L, nr, prec, monkeypatch):
    conf = conf_of(L, 57, [1.0, 0.2, 0, 0])
    mus = [0.05 + 0.01 * i for i in range(nr)]
    sols = []
    for tune, n in (("0", nr), ("r", nr), ("r", 1)):
        monkeypatch.setenv("NQ_TUNE", tune)
        with nq.Ctx(L) as ctx:
            g = nq.Gauge(ctx, lx=conf)
            src = [ctx.field(nq.SPINCOLOR, nq.LX, nq.source_lx(L, 95 + i)) for i in range(n)]
            sol = [ctx.field(nq.SPINCOLOR, nq.LX) for _ in range(n)]
            res = nq.tm_solve_eoprec_multi(ctx, g, 0.16, mus[:n], 1000, 1e-14, sol, src, prec=prec, anis=0.87)
            assert all(r["rc"] == nq.NQ_OK for r in res), res
            sols.append([f.download() for f in sol])
    for i in range(nr):
        assert np.array_equal(sols[0][i], sols[1][i]), i
    assert np.array_equal(sols[0][0], sols[2][0])


@pytest.mark.parametrize("L", [(10, 4, 2, 2), (4, 6, 4, 10), (8, 4, 4, 12)])
@pytest.mark.parametrize("theta", [[1.0, 0, 0, 0], [1.0, 0.3, -0.2, 0.5]])
def test_f16_solves_with_phases(L, theta):
    conf = conf_of(L, 52, theta)
    geo = orc.Geom(L)
    kappa, mus, n = 0.16, [0.05, 0.07, 0.09], 3
    src = [nq.source_lx(L, 70 + i) for i in range(n)]
    ref = [geo.tm_solve_eoprec(conf, kappa, mus[i], 20000, 1e-24, src[i])[0] for i in range(n)]
    ce, co = geo.split(conf)
    x = gauss_eo(geo.Vh, 8)
    with nq.Ctx(L) as ctx:
        g = nq.Gauge(ctx, lx=conf)
        fi, fo = ctx.field(nq.SPINCOLOR, nq.ODD, x), ctx.field(nq.SPINCOLOR, nq.EVEN)
        nq.tm_hop(ctx, g, fo, fi)
        assert rel_l2(fo.download(), geo.tm_hop(0, ce, co, x)) < 1e-14
        fs = [ctx.field(nq.SPINCOLOR, nq.LX, s) for s in src]
        fx = [ctx.field(nq.SPINCOLOR, nq.LX) for _ in src]
        for prec in ("f16", "f16h", "f32"):
            st = nq.tm_solve_eoprec(ctx, g, kappa, mus[0], 20000, 1e-24, fx[0], fs[0], prec=prec)
            assert st["rc"] == nq.NQ_OK
            assert rel_l2(fx[0].download(), ref[0]) < 1e-10, prec
            res = nq.tm_solve_eoprec_multi(ctx, g, kappa, mus, 20000, 1e-24, fx, fs, prec=prec)
            assert all(r["rc"] == nq.NQ_OK for r in res)
            for i in range(n):
                assert rel_l2(fx[i].download(), ref[i]) < 1e-10, (prec, i)


# every iteration count up to six: the shift vectors are updated in pairs of iterations,
# and the end comes on a first or a second one
@pytest.mark.parametrize("n", [1, 2, 3, 4, 5, 6])
def test_q2_multi_mass_iterates(n):
    L = (6, 4, 2, 4)
    conf = conf_of(L, 53, [1.0, 0, 0, 0])
    geo = orc.Geom(L)
    masses, residues = [0.1, 0.3, 0.9, 3.0], [1e-24, 1e-3, 1e-2, 1e-1]  # some stop on the way
    src = nq.source_lx(L, 80)
    ref = geo.tmQ2_cgm(conf, 0.12, masses, n, residues, src)[0]
    with nq.Ctx(L) as ctx:
        g = nq.Gauge(ctx, lx=conf)
        sols = [ctx.field(nq.SPINCOLOR, nq.LX) for _ in masses]
        st = nq.tmQ2_cgm(ctx, g, 0.12, masses, n, residues, sols, ctx.field(nq.SPINCOLOR, nq.LX, src))
        assert st["iters"] == n
        for k in range(4):
            assert rel_l2(sols[k].download(), ref[k]) < 1e-12, k



def test_persistent_hop_same_bits_large(monkeypatch):
    """262144 sites per parity, the smallest lattice of the persistent FP64 hop: the hop
    and a solve have the bits of the one-shot kernel."""
    L = (16, 32, 32, 32)
    conf = conf_of(L, 54, [1.0, 0, 0, 0])
    with nq.Ctx(L) as ctx:
        g = nq.Gauge(ctx, lx=conf)
        fi, fo = ctx.field(nq.SPINCOLOR, nq.ODD, gauss_eo(ctx.Vh, 9)), ctx.field(nq.SPINCOLOR, nq.EVEN)
        fs, fx = ctx.field(nq.SPINCOLOR, nq.LX, nq.source_lx(L, 11)), ctx.field(nq.SPINCOLOR, nq.LX)
        out = []
        for mode in ("1", "0"):
            monkeypatch.setenv("NQ_PERSIST", mode)
            nq.tm_hop(ctx, g, fo, fi)
            st = nq.tm_solve_eoprec(ctx, g, 0.16, 0.05, 1000, 1e-14, fx, fs)
            assert st["rc"] == nq.NQ_OK
            out.append((fo.download(), fx.download()))
        assert np.array_equal(out[0][0], out[1][0]) and np.array_equal(out[0][1], out[1][1])


# fewer sources per wavefront on lattices of few blocks: 256, 128 and 18 blocks, one partial
@pytest.mark.parametrize("L,nr", [((32, 16, 16, 16), 4), ((16, 16, 16, 16), 4), ((14, 10, 8, 8), 7), ((2, 4, 6, 2), 2)])
@pytest.mark.parametrize("prec", ["f64", "f32"])
def test_staggered_batch_same_bits_whatever_the_block(L, nr, prec, monkeypatch):
    out = {}
    for rb in (None, "1", "4", "6"):
        monkeypatch.delenv("NQ_ST_RB", raising=False)
        if rb:
            monkeypatch.setenv("NQ_ST_RB", rb)
        with nq.Ctx(L) as ctx:
            g = nq.Gauge(ctx, lx=st_conf(L, 7))
            src = [ctx.field(nq.COLOR, nq.EVEN, gauss_eo(np.prod(L) // 2, 70 + i, ncomp=3)) for i in range(nr)]
            sol = [[ctx.field(nq.COLOR, nq.EVEN) for _ in range(2)] for _ in src]
            res = nq.st_cgm(ctx, g, [0.09, 0.5], 2000, [1e-16, 1e-16], sol, src, prec=prec)
            assert all(r["rc"] == nq.NQ_OK for r in res), res
            out[rb] = np.stack([f.download() for s in sol for f in s])
    for rb in ("1", "4", "6"):
        assert np.array_equal(out[None], out[rb]), rb


def test_persistent_hop_against_oracle(monkeypatch):
    """32^4: 2048 blocks, at least twice the slots of 256 CUs that hold up to four workgroups
    of 48 KB of LDS in 160 KB, and too large to be split: the persistent FP64 hop, both
    parities against the oracle, and the one-shot kernel's bits."""
    L = (32, 32, 32, 32)
    conf = conf_of(L, 58, [1.0, 0, 0, 0])
    geo = orc.Geom(L)
    ce, co = geo.split(conf)
    x = gauss_eo(geo.Vh, 12)
    with nq.Ctx(L) as ctx:
        g = nq.Gauge(ctx, lx=conf)
        for out_par in (0, 1):
            fi, fo = ctx.field(nq.SPINCOLOR, 1 - out_par, x), ctx.field(nq.SPINCOLOR, out_par)
            monkeypatch.setenv("NQ_PERSIST", "1")
            nq.tm_hop(ctx, g, fo, fi)
            hop = fo.download()
            assert rel_l2(hop, geo.tm_hop(out_par, ce, co, x)) < 1e-14
            monkeypatch.setenv("NQ_PERSIST", "0")
            nq.tm_hop(ctx, g, fo, fi)
            assert np.array_equal(fo.download(), hop)


# links past the memory-side cache: the one-source hops with clover blocks are staged in LDS
# (NQ_LDS=0: they are not), and a batch runs the plain ones
@pytest.mark.parametrize("prec", ["f16", "f16h", "f32"])
def test_clover_with_streamed_links(prec, monkeypatch):
    L, kappa, mu, n = (40, 24, 24, 24), 0.13, 0.05, 3
    conf = conf_of(L, 59, [1.0, 0, 0, 0])
    with nq.Ctx(L) as ctx:
        g = nq.Gauge(ctx, lx=conf)
        cl = nq.Clover(ctx, g, 1.0)
        src = [ctx.field(nq.SPINCOLOR, nq.LX, nq.source_lx(L, 75 + i)) for i in range(n)]
        sol = [ctx.field(nq.SPINCOLOR, nq.LX) for _ in src]
        out = []
        for lds in ("1", "0"):
            monkeypatch.setenv("NQ_LDS", lds)
            st = nq.tmclov_solve_eoprec(ctx, g, cl, kappa, mu, 1000, 1e-14, sol[0], src[0], prec=prec)
            assert st["rc"] == nq.NQ_OK and st["rel_res_sq"] < 1e-14, st
            out.append(sol[0].download())
        assert np.array_equal(out[0], out[1])
        monkeypatch.delenv("NQ_LDS")
        res = nq.tmclov_solve_eoprec_multi(ctx, g, cl, kappa, mu, 1000, 1e-14, sol, src, prec=prec)
        assert all(r["rc"] == nq.NQ_OK and r["rel_res_sq"] < 1e-14 for r in res), res
        batch = [f.download() for f in sol]
        # |x - y| <= |(K K^+)^-1| (|r_x| + |r_y|) with |r| = 1e-7 |b| each; the smallest
        # eigenvalue of K K^+ is at least (2 kappa mu)^2 in units of the largest
        assert rel_l2(batch[0], out[0]) < 2e-7 / (2 * kappa * mu) ** 2
        one = [ctx.field(nq.SPINCOLOR, nq.LX)]
        nq.tmclov_solve_eoprec_multi(ctx, g, cl, kappa, mu, 1000, 1e-14, one, src[2:], prec=prec)
        assert np.array_equal(one[0].download(), batch[2])


# 110 blocks: staged from three right-hand sides up on 256 CUs; 40 blocks, from seven
@pytest.mark.parametrize("L,nr", [((28, 12, 12, 14), 3), ((10, 12, 12, 14), 7)])
@pytest.mark.parametrize("prec", ["f64", "f32", "f16"])
def test_staged_batch_same_bits_alone(L, nr, prec, monkeypatch):
    monkeypatch.setenv("NQ_TUNE", "0")  # the register-blocked kernel, also for FP16
    conf = conf_of(L, 60, [1.0, 0, 0, 0])
    with nq.Ctx(L) as ctx:
        g = nq.Gauge(ctx, lx=conf)
        src = [ctx.field(nq.SPINCOLOR, nq.LX, nq.source_lx(L, 65 + i)) for i in range(nr)]
        sol = [ctx.field(nq.SPINCOLOR, nq.LX) for _ in src]
        out = []
        for n in (nr, 1):
            res = nq.tm_solve_eoprec_multi(ctx, g, 0.16, [0.05] * n, 1000, 1e-14, sol[:n], src[:n], prec=prec)
            assert all(r["rc"] == nq.NQ_OK for r in res), res
            out.append(sol[0].download())
        assert np.array_equal(out[0], out[1])
