"""The work that users of this library have it do, as cases that can be timed.

Lattices are (T, X, Y, Z).  Gauge fields are U = exp(0.3 i H) per link with H Gaussian in
the algebra, as the benchmark makes them, with the antiperiodic time phase (twisted mass)
or the staggered and antiperiodic phases (staggered) applied.  kappa = 0.16 throughout,
as in the benchmark and the tests.  Fields stay on the device between calls, as a user's
program keeps them; the host-buffer calls take and return host arrays.
"""
import math

import numpy as np
import torch
from torch.utils._pytree import tree_map

import nissa_amd as nq

DEV = "cuda" if torch.cuda.is_available() else "cpu"
KAPPA = 0.16


# ---------------------------------------------------------------- the cases
def listed():
    return [
        # one Dslash on a lattice of unit-test size: the cost of one call
        _case("hop_f64_8c8", "hop", (8, 8, 8, 8)),
        # K K^+ as an HMC or a caller's own solver applies it, on uneven extents (5040 sites
        # a parity: no multiple of the wavefront)
        _case("kernsq_f64_12x6x10x14", "kernsq", (12, 6, 10, 14), mu=0.05),
        # the same at the size of the benchmark's FP64 Dslash
        _case("kernsq_f64_24c48", "kernsq", (48, 24, 24, 24), mu=0.005),
        # FP64 eo solve on a small lattice (tests, tuning runs): bound by launches and latency
        _case("solve_f64_8c16", "solve", (16, 8, 8, 8), prec="f64", mu=0.01, residue=1e-24),
        # the benchmark's headline: FP16-inner eo solve at 32^3x64
        _case("solve_f16_32c64", "solve", (64, 32, 32, 32), prec="f16", mu=0.003, residue=1e-20),
        # the same with FP16 links on a middle lattice
        _case("solve_f16h_24c48", "solve", (48, 24, 24, 24), prec="f16h", mu=0.005, residue=1e-20),
        # a propagator: 12 spin-colour point sources in one batch (the serving mix's middle volume)
        _case("propagator_f16_24c48", "multi", (48, 24, 24, 24), prec="f16", mu=0.005, residue=1e-20, nsrc=12),
        # a propagator on the serving mix's most frequent volume
        _case("propagator_f16_16c32", "multi", (32, 16, 16, 16), prec="f16", mu=0.01, residue=1e-20, nsrc=12),
        # twisted-clover solve with FP16 inner iterations
        _case("clover_f16_24c48", "clover", (48, 24, 24, 24), prec="f16", mu=0.003, residue=1e-20, csw=1.0),
        # rational approximation of the staggered determinant (RHMC action or heat bath):
        # one multi-shift solve over its poles for a few pseudofermions
        _case("ratsum_f32_24c48", "ratsum", (48, 24, 24, 24), prec="f32", residue=1e-20, nsrc=4, nshift=12),
        # multi-mass solve on Q^2 over the whole lattice (twisted-mass RHMC, several masses at once)
        _case("q2cgm_f64_16c32", "q2cgm", (32, 16, 16, 16), prec="f64", residue=1e-20, nshift=4, mu=0.01),
        # the drop-in call on the caller's host buffers: source up, FP64 solve, solution down
        _case("host_solve_f64_16c32", "host", (32, 16, 16, 16), prec="f64", mu=0.01, residue=1e-24),
    ]


def _case(name, family, L, prec="f64", mu=0.0, residue=1e-20, nsrc=1, nshift=0, csw=0.0):
    c = {"family": family, "T": L[0], "X": L[1], "Y": L[2], "Z": L[3], "prec": prec, "mu": mu, "residue": residue,
         "nsrc": nsrc, "nshift": nshift, "csw": csw}
    if name:
        c["name"] = name
    return c


# largest volume (sites) of a drawn case, so that none costs more than the largest listed one
_MOST = {"hop": 2 ** 21, "kernsq": 2 ** 21, "solve": 2 ** 21, "multi": 48 * 24 ** 3, "clover": 48 * 24 ** 3,
         "ratsum": 48 * 24 ** 3, "q2cgm": 32 * 16 ** 3, "host": 32 * 16 ** 3}


def draw(rng):
    family = rng.choice(sorted(_MOST))
    # the volume spread over its logarithm, the extents even (as the lattice has to be) and
    # otherwise free
    most = _MOST[family]
    while True:
        v = 2.0 ** rng.uniform(10.0, math.log2(most))
        L = []
        for k in range(3):
            s = (v / 2.0) ** 0.25 * 2.0 ** rng.uniform(-0.4, 0.4)
            L.append(max(4, min(32, 2 * round(s / 2))))
        t = 2 * round(v / (L[0] * L[1] * L[2]) / 2)
        if 4 <= t <= 64 and t * L[0] * L[1] * L[2] <= most:
            break
    L = (t, L[0], L[1], L[2])
    mu = round(rng.uniform(0.003, 0.02), 4)
    if family in ("hop", "kernsq"):
        return _case("", family, L, mu=mu if family == "kernsq" else 0.0)
    if family in ("solve", "clover"):
        prec = rng.choice(["f64", "f32", "f16", "f16h"])
        residue = rng.choice([1e-20, 1e-22])
        return _case("", family, L, prec=prec, mu=mu, residue=residue, csw=rng.choice([0.5, 1.0, 1.3]) if family == "clover" else 0.0)
    if family == "multi":
        return _case("", family, L, prec=rng.choice(["f32", "f16", "f16", "f16h"]), mu=mu, residue=1e-20,
                     nsrc=rng.randint(2, 12))
    if family == "ratsum":
        return _case("", family, L, prec=rng.choice(["f64", "f32"]), residue=1e-20, nsrc=rng.randint(1, 4),
                     nshift=rng.randint(4, 12))
    if family == "q2cgm":
        return _case("", family, L, residue=1e-20, nshift=rng.randint(2, 4), mu=mu)
    return _case("", family, L, prec=rng.choice(["f64", "f16"]), mu=mu, residue=rng.choice([1e-20, 1e-22]))


def _dims(c):
    return c["T"], c["X"], c["Y"], c["Z"]


def _poles(c):
    """Poles and weights of the rational sum: m^2 + 10^(-4 + 5k/(n-1)), m = 0.0025."""
    n = c["nshift"]
    p = [0.0025 ** 2 + 10 ** (-4 + 5 * k / max(1, n - 1)) for k in range(n)]
    return p, [0.3 * math.sqrt(x) for x in p]


def _masses(c):
    return [c["mu"] * 2 ** k for k in range(c["nshift"])]


# ---------------------------------------------------------------- inputs
def _randn(shape, seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(seed)
    return torch.randn(*shape, dtype=torch.float64, device=DEV, generator=g)


def _mul3(a, b):
    return sum(a[..., :, k, None] * b[..., None, k, :] for k in range(3))


def _gauge(c, seed):
    """Links (T, X, Y, Z, mu, 3, 3) with the phases of the case's fermions."""
    L = _dims(c)
    V = math.prod(L)
    U = torch.empty((V, 4, 3, 3), dtype=torch.complex128, device=DEV)
    for mu in range(4):
        a = torch.view_as_complex(_randn((V, 3, 3, 2), 1000 * seed + mu)) * math.sqrt(0.5)
        h = (a + a.mH) * math.sqrt(0.5)
        tr = (h[:, 0, 0] + h[:, 1, 1] + h[:, 2, 2]) / 3
        for k in range(3):
            h[:, k, k] -= tr
        h *= 0.3j
        # exp by its series (|h| stays below 3), rows made orthonormal to rounding
        term, u = h.clone(), h.clone()
        for k in range(3):
            u[:, k, k] += 1
        for n in range(2, 30):
            term = _mul3(term, h) / n
            u += term
        r0 = u[:, 0] / u[:, 0].abs().square().sum(-1, keepdim=True).sqrt()
        r1 = u[:, 1] - (r0.conj() * u[:, 1]).sum(-1, keepdim=True) * r0
        r1 = r1 / r1.abs().square().sum(-1, keepdim=True).sqrt()
        U[:, mu, 0], U[:, mu, 1] = r0, r1
        for j in range(3):
            x, y = (j + 1) % 3, (j + 2) % 3
            U[:, mu, 2, j] = (r0[:, x] * r1[:, y] - r0[:, y] * r1[:, x]).conj()
    U = U.view(*L, 4, 3, 3)
    staggered = c["family"] == "ratsum"
    if staggered:
        n = torch.arange(64, device=DEV)
        sign = [None] * 4  # eta_t = 1, eta_x = (-1)^t, eta_y = (-1)^(t+x), eta_z = (-1)^(t+x+y)
        t, x, y = n[:L[0]].view(-1, 1, 1, 1), n[:L[1]].view(1, -1, 1, 1), n[:L[2]].view(1, 1, -1, 1)
        sign[1], sign[2], sign[3] = t, t + x, t + x + y
        for mu in (1, 2, 3):
            U[..., mu, :, :] *= (1 - 2 * (sign[mu] % 2)).to(torch.float64)[..., None, None]
    ph = math.pi / L[0] * (-1 if staggered else 1)
    U[..., 0, :, :] *= complex(math.cos(ph), math.sin(ph))
    return U


def _sources(c, seed):
    """The case's right-hand sides on the whole lattice, (T, X, Y, Z, spin, colour) or (..., colour)."""
    L = _dims(c)
    V = math.prod(L)
    if c["family"] == "multi":  # spin-colour point sources at one site
        site, out = (7919 * seed + 13) % V, []
        for k in range(c["nsrc"]):
            s = torch.zeros((V, 12), dtype=torch.complex128, device=DEV)
            s[site, k] = 1
            out.append(s.view(*L, 4, 3))
        return out
    colour = c["family"] == "ratsum"
    shape = (*L, 3) if colour else (*L, 4, 3)
    out = [torch.view_as_complex(_randn((*shape, 2), 1000 * seed + 500 + k)) * math.sqrt(0.5) for k in range(c["nsrc"])]
    par = _parity(L)
    if colour or c["family"] == "hop":  # even sites of the staggered source; odd sites into the even hop
        keep = (par == 0) if colour else (par == 1)
        out = [s * keep.view(*L, *([1] * (s.dim() - 4))) for s in out]
    if c["family"] == "kernsq":
        out = [s * (par == 1).view(*L, 1, 1) for s in out]
    return out


def _parity(L):
    n = [torch.arange(x, device=DEV) for x in L]
    return (n[0].view(-1, 1, 1, 1) + n[1].view(1, -1, 1, 1) + n[2].view(1, 1, -1, 1) + n[3].view(1, 1, 1, -1)) % 2


def _half(x, L, par):
    """The sites of one parity in lx order, which is the library's eo order."""
    return x.reshape(math.prod(L), *x.shape[4:])[(_parity(L) == par).view(-1)]


def _host(x):
    return torch.view_as_real(x.contiguous()).cpu().numpy()


# ---------------------------------------------------------------- outputs
class FieldTensor(torch.Tensor):
    """A field of the library as a tensor: it stays on the device where the library keeps it,
    and its values are read with download() by whatever looks at them."""

    @staticmethod
    def __new__(cls, field):
        return torch.Tensor._make_wrapper_subclass(cls, field.shape, dtype=torch.float64)

    def __init__(self, field):
        self.field = field

    @classmethod
    def __torch_dispatch__(cls, func, types, args=(), kwargs=None):
        args, kwargs = tree_map(lambda a: torch.from_numpy(a.field.download()) if isinstance(a, cls) else a,
                                (tuple(args), kwargs or {}))
        return func(*args, **kwargs)


# ---------------------------------------------------------------- prepare and run
def prepare(case, seed):
    c = dict(case)
    L, fam = _dims(c), c["family"]
    U = _gauge(c, seed)
    s = {"case": c, "ctx": nq.Ctx(L)}
    ctx = s["ctx"]
    s["g"] = ctx.gauge_eo(_host(_half(U, L, 0)), _host(_half(U, L, 1)))
    del U
    src = _sources(c, seed)
    if fam in ("hop", "kernsq"):
        s["in"] = ctx.field(nq.SPINCOLOR, nq.ODD, _host(_half(src[0], L, 1)))
        s["out"] = [ctx.field(nq.SPINCOLOR, nq.EVEN if fam == "hop" else nq.ODD)]
    elif fam == "ratsum":
        s["in"] = [ctx.field(nq.COLOR, nq.EVEN, _host(_half(x, L, 0))) for x in src]
        s["out"] = [ctx.field(nq.COLOR, nq.EVEN) for _ in src]
    elif fam == "host":
        s["in"] = _host(src[0]).reshape(-1, 4, 3, 2)
    else:
        s["in"] = [ctx.field(nq.SPINCOLOR, nq.LX, _host(x)) for x in src]
        s["out"] = [ctx.field(nq.SPINCOLOR, nq.LX) for _ in range(c["nshift"] if fam == "q2cgm" else c["nsrc"])]
        if fam == "clover":
            s["cl"] = nq.Clover(ctx, s["g"], c["csw"])
    return s


def run(s):
    c, ctx, g = s["case"], s["ctx"], s["g"]
    fam, mu, res, prec = c["family"], c["mu"], c["residue"], c["prec"]
    if fam == "hop":
        nq.tm_hop(ctx, g, s["out"][0], s["in"])
    elif fam == "kernsq":
        nq.tm_kern_square(ctx, g, KAPPA, mu, s["out"][0], s["in"])
    elif fam == "solve":
        nq.tm_solve_eoprec(ctx, g, KAPPA, mu, 100000, res, s["out"][0], s["in"][0], prec=prec)
    elif fam == "multi":
        nq.tm_solve_eoprec_multi(ctx, g, KAPPA, [mu] * c["nsrc"], 100000, res, s["out"], s["in"], prec=prec)
    elif fam == "clover":
        nq.tmclov_solve_eoprec(ctx, g, s["cl"], KAPPA, mu, 100000, res, s["out"][0], s["in"][0], prec=prec)
    elif fam == "ratsum":
        poles, weights = _poles(c)
        nq.st_cgm_rat_sum(ctx, g, 0.5, poles, weights, 100000, res, s["out"], s["in"], prec=prec)
    elif fam == "q2cgm":
        m = _masses(c)
        nq.tmQ2_cgm(ctx, g, KAPPA, m, 100000, [res] * len(m), s["out"], s["in"][0])
    else:
        x, _ = nq.tm_solve_eoprec_host(ctx, g, KAPPA, mu, 100000, res, s["in"], prec=prec)
        return x
    return [FieldTensor(f) for f in s["out"]]


# ---------------------------------------------------------------- compulsory work
_LINK = {"f64": 1152, "f32": 576, "f16": 384, "f16h": 192}  # the eight links of a site, as each precision holds them
_SPIN = {"f64": 192, "f32": 96, "f16": 52, "f16h": 52}


def work(case):
    """Each operator of the iteration reads its links and input once and writes its output
    once; a solve takes about as many iterations per decade of the residue as the benchmark's
    (3.2 twisted mass, 2.7 clover, 9.8 on Q^2, 28 staggered)."""
    c = case
    vh = math.prod(_dims(c)) / 2
    fam, pr = c["family"], c["prec"]
    lk, sp = _LINK[pr], _SPIN[pr]
    hop = lk + 2 * sp
    dec = -math.log10(c["residue"])
    if fam == "hop":
        return {"bytes": vh * hop, "flops": vh * 1320}
    if fam == "kernsq":
        return {"bytes": vh * (4 * hop + 2 * sp), "flops": vh * 4 * 1400}
    if fam in ("solve", "host", "clover", "multi"):
        xr = 192 if pr == "f64" else 96
        it = dec * (2.7 if fam == "clover" else 3.2)
        n = c["nsrc"]
        blk = 0 if fam != "clover" else 2 * (72 + 36) * {"f64": 16, "f32": 8}.get(pr, 4)
        per = 4 * lk + blk + n * (4 * 2 * sp + 2 * sp + 4 * xr + 3 * sp)
        io = 2 * vh * 2 * 192 * n  # source in, solution out
        return {"bytes": it * vh * per + io, "flops": it * vh * n * (4 * 1400 + 200 + (4 * 500 if blk else 0))}
    if fam == "q2cgm":
        it, n = dec * 9.8, c["nshift"]
        return {"bytes": it * 2 * vh * (2 * (1152 + 3 * 192) + 192 * (4 + 3 * n)), "flops": it * 2 * vh * (2 * 1400 + 100 * n)}
    it, n, k = dec * 28, c["nsrc"], c["nshift"]
    st = 48 if pr == "f64" else 24
    # about a third of the shifts of a rational approximation still run on average
    return {"bytes": it * vh * (2 * (1152 if pr == "f64" else 576) + n * st * (8 + 3 * k / 3)),
            "flops": it * vh * n * (2 * 570 + 24 * k / 3)}


# ---------------------------------------------------------------- the results in 64 bits
# gamma_mu = [[0, B], [B^+, 0]] for t, x, y, z: B as (column, phase) per row
_B = [((0, -1), (1, -1)), ((1, -1j), (0, -1j)), ((1, -1), (0, 1)), ((0, -1j), (1, 1j))]


def _spin2(rows, v):
    return torch.stack([ph * v[..., col, :] for col, ph in rows], dim=-2)


def _dagger2(rows):
    out = [None, None]
    for r, (col, ph) in enumerate(rows):
        out[col] = (r, complex(ph).conjugate())
    return out


def _matvec(u, h):
    """u (..., 3, 3) on each colour vector of h (..., spins, 3)."""
    return sum(u[..., None, :, k] * h[..., k, None] for k in range(3))


def _hop(U, psi):
    """sum_mu (1 - g_mu) U_mu(x) psi(x+mu) + (1 + g_mu) U_mu(x-mu)^+ psi(x-mu)."""
    out = torch.zeros_like(psi)
    for mu in range(4):
        B, C = _B[mu], _dagger2(_B[mu])
        u = U[..., mu, :, :]
        h = torch.roll(psi[..., :2, :] - _spin2(B, psi[..., 2:, :]), -1, mu)
        f = _matvec(u, h)
        out[..., :2, :] += f
        out[..., 2:, :] -= _spin2(C, f)
        h = psi[..., :2, :] + _spin2(B, psi[..., 2:, :])
        f = torch.roll(_matvec(u.mH, h), 1, mu)
        out[..., :2, :] += f
        out[..., 2:, :] += _spin2(C, f)
    return out


def _g5(psi):
    out = psi.clone()
    out[..., 2:, :] *= -1
    return out


def _diag(psi, up, lo):
    return torch.cat([psi[..., :2, :] * up, psi[..., 2:, :] * lo], dim=-2)


def _kern(U, mu, psi):
    """K(mu) = g5 (D_oo - 1/4 H D_ee^-1 H)."""
    a, b = complex(1 / (2 * KAPPA), mu), complex(1 / (2 * KAPPA), -mu)
    e = _diag(_hop(U, psi), 1 / a, 1 / b)
    return _g5(_diag(psi, a, b) - 0.25 * _hop(U, e))


def _clover(U, csw):
    """F (plane, ..., 3, 3): the clover average (Q - Q^+)/4 of each plane."""
    def at(x, mu, n):
        return torch.roll(x, -n, mu)

    out = []
    for mu in range(4):
        for nu in range(mu + 1, 4):
            a, b = U[..., mu, :, :], U[..., nu, :, :]
            bd, ad = at(b, mu, -1), at(a, mu, -1)  # links at x - mu
            bf, af = at(b, nu, -1), at(a, nu, -1)  # links at x - nu
            q = _mul3(_mul3(a, at(b, mu, 1)), _mul3(b, at(a, nu, 1)).mH)
            q = q + _mul3(_mul3(b, at(ad, nu, 1).mH), _mul3(bd.mH, ad))
            q = q + _mul3(_mul3(at(bd, nu, -1), ad).mH, _mul3(at(ad, nu, -1), bf))
            q = q + _mul3(_mul3(bf.mH, af), _mul3(at(bf, mu, 1), a.mH))
            out.append((mu, nu, (q - q.mH) * (0.25 * -csw / 4)))
    return out


def _gamma(mu, psi):
    return torch.cat([_spin2(_B[mu], psi[..., 2:, :]), _spin2(_dagger2(_B[mu]), psi[..., :2, :])], dim=-2)


def _dirac(U, mu, psi, clover=()):
    """D = 1/(2 kappa) + i mu g5 + clover - H/2."""
    a, b = complex(1 / (2 * KAPPA), mu), complex(1 / (2 * KAPPA), -mu)
    out = _diag(psi, a, b) - 0.5 * _hop(U, psi)
    for m, n, f in clover:
        out += _gamma(m, _gamma(n, _matvec(f, psi)))
    return out


def _dot(a, b):
    return torch.vdot(a.reshape(-1), b.reshape(-1)).real.item()


def _cg(A, b, drop):
    """x with |b - A x| <= drop |b|, A hermitian and positive."""
    x, r = torch.zeros_like(b), b.clone()
    p, rr = r.clone(), _dot(b, b)
    stop, n = rr * drop * drop, 0
    while rr > stop and n < 20000:
        q = A(p)
        al = rr / _dot(p, q)
        x += al * p
        r -= al * q
        new = _dot(r, r)
        p = r + (new / rr) * p
        rr, n = new, n + 1
    return x


def _solve(A, b):
    """A x = b to rounding: a solve, and one on what it left."""
    x = _cg(A, b, 1e-12)
    return x + _cg(A, b - A(x), 1e-5)


def _solve_dirac(U, mu, b, clover=()):
    def adj(v):  # D(mu)^+ = g5 D(-mu) g5
        return _g5(_dirac(U, mu, _g5(v), clover)) - _diag(v, 2j * mu, -2j * mu)

    y = _solve(lambda v: _dirac(U, mu, adj(v), clover), b)
    return adj(y)


def _st_hop(U, v):
    """sum_mu U_mu(x) v(x+mu) - U_mu(x-mu)^+ v(x-mu)."""
    out = torch.zeros_like(v)
    for mu in range(4):
        u = U[..., mu, :, :]
        out += _matvec(u, torch.roll(v, -1, mu)[..., None, :])[..., 0, :]
        out -= torch.roll(_matvec(u.mH, v[..., None, :])[..., 0, :], 1, mu)
    return out


def _out(x, L, par=None):
    x = x.reshape(math.prod(L), *x.shape[4:]) if par is None else _half(x, L, par)
    return torch.view_as_real(x.contiguous()).cpu()


def exact(case, seed):
    c = dict(case)
    L, fam = _dims(c), c["family"]
    U, src = _gauge(c, seed), _sources(c, seed)
    if fam == "hop":
        return [_out(_hop(U, src[0]), L, 0)]
    if fam == "kernsq":
        return [_out(_kern(U, c["mu"], _kern(U, -c["mu"], src[0])), L, 1)]
    if fam == "solve":
        return [_out(_solve_dirac(U, c["mu"], src[0]), L)]
    if fam == "clover":
        return [_out(_solve_dirac(U, c["mu"], src[0], _clover(U, c["csw"])), L)]
    if fam == "host":
        return _out(_solve_dirac(U, c["mu"], src[0]), L).numpy()
    if fam == "multi":  # the first sources: all of them take longer than the checks are worth
        return [_out(_solve_dirac(U, c["mu"], b), L) if k < 2 else None for k, b in enumerate(src)]
    if fam == "q2cgm":
        def q2(v):
            return _g5(_dirac(U, 0.0, _g5(_dirac(U, 0.0, v))))

        return [_out(_solve(lambda v: q2(v) + m * m * v, src[0]), L) for m in _masses(c)]
    poles, weights = _poles(c)
    out = []
    for k, b in enumerate(src):
        if k > 0:
            out.append(None)
            continue
        x = 0.5 * b
        for p, w in zip(poles, weights):
            x = x + w * _solve(lambda v: p * v - 0.25 * _st_hop(U, _st_hop(U, v)), b)
        out.append(_out(x, L, 0))
    return out
