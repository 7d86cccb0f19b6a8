"""The z tile of the site order: it moves sites and not the arithmetic of a site, whatever
its length; and a choice of the other tiles is cached for the z tile it was timed with."""
import numpy as np
import pytest

import nissa_amd as nq
from helpers import gauss_eo, rel_l2, tm_conf
from oracle import oracle as orc

pytestmark = pytest.mark.gpu


def test_cached_tiles_belong_to_a_z_tile(tmp_path, monkeypatch):
    L = (32, 16, 32, 32)
    cache = tmp_path / "site_tiles.txt"
    monkeypatch.setenv("NQ_TUNE_CACHE", str(cache))
    for e in ("NQ_TTILE", "NQ_XYTILE", "NQ_TUNE_TILES", "NQ_ZTILE"):
        monkeypatch.delenv(e, raising=False)
    # lines from before the order had a z tile; the tuner never takes a t tile of 2
    old = "".join(f"{a} 32 16 32 32 2 1 1 90.0 30.0\n" for a in ("gfx950", "unknown"))
    cache.write_text(old)
    tiles = {}
    for z in (2, 4):
        monkeypatch.setenv("NQ_ZTILE", str(z))
        with nq.Ctx(L) as ctx:
            tiles[z] = ctx.site_tiles()
    lines = [l.split() for l in cache.read_text()[len(old):].splitlines()]
    assert [int(l[-1]) for l in lines] == [2, 4], lines
    for l in lines:
        assert tuple(int(v) for v in l[5:8]) == tiles[int(l[-1])] != (2, 1, 1)
    monkeypatch.setenv("NQ_ZTILE", "2")
    with nq.Ctx(L) as ctx:
        assert ctx.site_tiles() == tiles[2]
    assert len(cache.read_text()[len(old):].splitlines()) == 2


# no cells, a cell of four rows, one that shrinks to two of ten rows, one longer than the extent
@pytest.mark.parametrize("L,z", [((8, 8, 4, 8), 1), ((8, 8, 4, 8), 4), ((4, 6, 4, 10), 8), ((8, 4, 4, 4), 16)])
def test_z_tiles(L, z, monkeypatch):
    conf = tm_conf(L, 21)
    geo = orc.Geom(L)
    ce, co = geo.split(conf)
    x = gauss_eo(geo.Vh, 22)
    src = nq.source_lx(L, 23)
    ref = geo.tm_solve_eoprec(conf, 0.16, 0.05, 20000, 1e-24, src)[0]
    hops = []
    for tile in (None, str(z)):
        monkeypatch.delenv("NQ_ZTILE", raising=False)
        if tile:
            monkeypatch.setenv("NQ_ZTILE", tile)
        with nq.Ctx(L) as ctx:
            g = nq.Gauge(ctx, lx=conf)
            for out_par in (0, 1):
                fi, fo = ctx.field(nq.SPINCOLOR, 1 - out_par, x), ctx.field(nq.SPINCOLOR, out_par)
                nq.tm_hop(ctx, g, fo, fi)
                hops.append(fo.download())
                assert rel_l2(hops[-1], geo.tm_hop(out_par, ce, co, x)) < 1e-14
            fs = [ctx.field(nq.SPINCOLOR, nq.LX, src) for _ in range(3)]
            fx = [ctx.field(nq.SPINCOLOR, nq.LX) for _ in fs]
            for prec in ("f64", "f16"):  # one source, and the batched kernels
                assert nq.tm_solve_eoprec(ctx, g, 0.16, 0.05, 20000, 1e-24, fx[0], fs[0], prec=prec)["rc"] == nq.NQ_OK
                assert rel_l2(fx[0].download(), ref) < 1e-10
                res = nq.tm_solve_eoprec_multi(ctx, g, 0.16, [0.05] * 3, 20000, 1e-24, fx, fs, prec=prec)
                assert all(r["rc"] == nq.NQ_OK for r in res)
                assert rel_l2(fx[2].download(), ref) < 1e-10
    assert np.array_equal(hops[0], hops[2]) and np.array_equal(hops[1], hops[3])
