"""The work that is timed: what a lattice-QCD program has this library do.

Every case goes through the public entry points (the C interface, by way of
pyqphix.api), with host arrays in MILC's raw order where a caller of that
interface passes them.  Kinds of work:

  operator    v <- D v on the whole lattice, `applications` times with the
              vectors kept on the device, the last one read back (residual
              checks, eigensolvers, polynomial filters)
  solve       one staggered solve of MILC's f_meas / spectrum calls: source in,
              CG (FP64, or mixed precision), solution out; the links are a
              handle that the program keeps for many sources
  handover    the same as MILC calls it on links it smeared itself: the four
              raw link arrays are handed over first, and dropped afterwards
  shifts      one multi-shift solve of a rational approximation (RHMC)
  sources     several sources x several shifts at once (batched mixed solver)
  refresh     fermion links rebuilt from a new gauge field, then the operator
  force       one Symanzik gauge-force step as MILC calls it: links and momenta
              in, momenta out
  trajectory  pure-gauge molecular dynamics, links and momenta in and out
  outer       fermion-force outer products of the solutions kept on the device
"""
import os
import sys
import weakref

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.getcwd(), "milc-qphix_amd"))
from pyqphix import api as A  # noqa: E402
from pyqphix import fields as F  # noqa: E402
from pyqphix import lib as Q  # noqa: E402

NP = {"D": np.float64, "F": np.float32}
ASQTAD = (5.0 / 8, -1.0 / 24, 1.0 / 16, 1.0 / 64, 1.0 / 384, -1.0 / 16)  # MILC's order, u0 = 1
NAIK_EPS = 0.0
OMELYAN = 0.1931833275037836


def _case(kind, dims, prec="D", **more):
    return {"kind": kind, "nx": dims[0], "ny": dims[1], "nz": dims[2], "nt": dims[3], "prec": prec, **more}


def listed():
    def named(name, *a, **k):
        return {"name": name, **_case(*a, **k)}

    return [
        # the smallest calls: both halves of D v on a test-sized lattice (latency)
        named("operator_8x8x8x8_D", "operator", (8, 8, 8, 8), links="su3", applications=1),
        # an eigensolver's or filter's run of applications, single precision, ragged extents
        named("operator_20x28x24x36_F", "operator", (20, 28, 24, 36), "F", links="su3", applications=8),
        # the same in double precision on the benchmark's lattice, HISQ links (18-real Naik)
        named("operator_32x32x32x32_D", "operator", (32, 32, 32, 32), links="hisq", applications=8),
        # a valence solve on a small ensemble, HISQ links
        named("solve_12x12x12x20_D", "solve", (12, 12, 12, 20), links="hisq", method="cg", mass=0.05),
        # the benchmark's FP64 solve
        named("solve_32x32x32x32_D", "solve", (32, 32, 32, 32), links="su3", method="cg", mass=0.02),
        # MILC hands its links over and solves once, mixed precision
        named("handover_24x24x24x32_mixed", "handover", (24, 24, 24, 32), links="su3", method="mixed", mass=0.05),
        # one RHMC solve of a molecular-dynamics step on a small ensemble
        named("shifts_16x16x16x32_D", "shifts", (16, 16, 16, 32), links="hisq", nshift=9, low=1e-3),
        # sources of one configuration solved together for all shifts
        named("sources_24x24x24x32_D", "sources", (24, 24, 24, 32), links="su3", nshift=7, nrhs=8, low=5e-4),
        # after each gauge update of HISQ molecular dynamics
        named("refresh_24x24x24x24_D", "refresh", (24, 24, 24, 24), links="hisq"),
        # the fermion force's outer products of a rational approximation's solutions
        named("outer_16x20x20x24_D", "outer", (16, 20, 20, 24), links="hisq", terms=9),
        # MILC's force call on a ragged lattice, and a quenched trajectory
        named("force_16x20x12x24_F", "force", (16, 20, 12, 24), "F", eps=0.02),
        named("trajectory_24x24x24x24_D", "trajectory", (24, 24, 24, 24), eps=0.02, nsteps=6),
    ]


# most of (sites x work) that a draw of each kind may have, below the listed ones' largest
_MOST_SITES = {"operator": 32 ** 4, "solve": 24 ** 3 * 32, "handover": 24 ** 3 * 24, "shifts": 24 ** 4,
               "sources": 16 ** 3 * 24, "refresh": 24 ** 4, "force": 28 ** 4, "trajectory": 24 ** 4,
               "outer": 24 ** 4}


def _draw_dims(rng, most):
    """Extents of 4..40 in steps of 4, the volume spread over its logarithm."""
    lo = 8 ** 4
    want = lo * (most / lo) ** rng.random()
    side = want ** 0.25
    for _ in range(1000):
        d = [max(4, min(40, 4 * round(side * rng.uniform(0.6, 1.6) / 4))) for _ in range(4)]
        v = d[0] * d[1] * d[2] * d[3]
        if max(lo // 2, 0.6 * want) <= v <= min(most, 1.6 * want):
            return d
    return [8, 8, 8, 8]


def draw(rng):
    kind = rng.choice(["operator", "operator", "solve", "solve", "handover", "shifts", "sources", "refresh", "force", "trajectory",
                       "outer"])
    dims = _draw_dims(rng, _MOST_SITES[kind])
    links = rng.choice(["su3", "hisq"])
    if kind == "operator":
        return _case(kind, dims, rng.choice("DF"), links=rng.choice(["su3", "hisq", "asqtad"]), applications=rng.randint(1, 8))
    if kind == "solve":
        return _case(kind, dims, links=links, method=rng.choice(["cg", "mixed", "mixed16"]), mass=round(rng.uniform(0.03, 0.2), 3))
    if kind == "handover":
        return _case(kind, dims, links=links, method=rng.choice(["cg", "mixed"]), mass=round(rng.uniform(0.04, 0.2), 3))
    if kind == "shifts":
        return _case(kind, dims, links=links, nshift=rng.randint(3, 14), low=10 ** rng.uniform(-3, -2))
    if kind == "sources":
        return _case(kind, dims, links=links, nshift=rng.randint(2, 8), nrhs=rng.randint(2, 8), low=10 ** rng.uniform(-3, -2))
    if kind == "refresh":
        return _case(kind, dims, rng.choice("DF"), links=rng.choice(["hisq", "asqtad"]))
    if kind == "force":
        return _case(kind, dims, rng.choice("DF"), eps=round(rng.uniform(0.005, 0.05), 4))
    if kind == "trajectory":
        return _case(kind, dims, eps=round(rng.uniform(0.01, 0.03), 4), nsteps=rng.randint(1, 6))
    return _case("outer", dims, rng.choice("DF"), links=links, terms=rng.randint(1, 9))


# ---------------------------------------------------------------- geometry
class Geo:
    """Raw (even sites first) indices of a lattice, as tensors on the GPU."""

    def __init__(self, dims):
        self.dims = tuple(dims)
        self.V = dims[0] * dims[1] * dims[2] * dims[3]
        self.vh = self.V // 2
        lex = torch.arange(self.V, device="cuda")
        c = []
        for n in dims:
            c.append(lex % n)
            lex = lex // n
        raw = self._raw(c)
        self.c = [torch.empty_like(k) for k in c]
        for k in range(4):
            self.c[k][raw] = c[k]

    def _raw(self, c):
        lex = c[0] + self.dims[0] * (c[1] + self.dims[1] * (c[2] + self.dims[2] * c[3]))
        return ((c[0] + c[1] + c[2] + c[3]) & 1) * self.vh + torch.div(lex, 2, rounding_mode="floor")

    def nbr(self, mu, hop):
        """Raw index of x + hop mu for every raw site x."""
        c = list(self.c)
        c[mu] = (c[mu] + hop) % self.dims[mu]
        return self._raw(c)

    def sign(self, mu, hop):
        """MILC's staggered phase of a link times its antiperiodic time boundary."""
        x, y, t = self.c[0], self.c[1], self.c[3]
        e = [t, t + x, t + x + y, torch.zeros_like(t)][mu] & 1
        if mu == 3:
            e = e ^ (t + hop >= self.dims[3]).long()
        return 1.0 - 2.0 * e.double()


def _dag(u):
    return u.conj().transpose(-1, -2)


def _mm(a, b):
    """3x3 products, elementwise in 64 bits."""
    r = a[..., :, 0:1] * b[..., 0:1, :]
    for k in (1, 2):
        r = r + a[..., :, k:k + 1] * b[..., k:k + 1, :]
    return r


def _mv(a, v):
    return a[..., 0] * v[..., 0:1] + a[..., 1] * v[..., 1:2] + a[..., 2] * v[..., 2:3]


# ---------------------------------------------------------------- inputs
def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed) * 7919 + 17)
    return g


def _gauss(g, *shape):
    return torch.complex(torch.randn(*shape, generator=g, device="cuda", dtype=torch.float64),
                         torch.randn(*shape, generator=g, device="cuda", dtype=torch.float64))


def _algebra(g, n):
    """n Gaussian traceless anti-Hermitian matrices."""
    z = _gauss(g, n, 3, 3)
    a = 0.5 * (z - _dag(z))
    tr = (a[:, 0, 0] + a[:, 1, 1] + a[:, 2, 2]) / 3.0
    return a - tr[:, None, None] * torch.eye(3, dtype=torch.complex128, device="cuda")


def _expm(a):
    """Matrix exponential by scaling and squaring of a Taylor series."""
    e = torch.eye(3, dtype=torch.complex128, device="cuda").expand_as(a)
    s = a / 64.0
    r = e.clone()
    for k in range(12, 0, -1):
        r = e + _mm(s, r) / k
    for _ in range(6):
        r = _mm(r, r)
    return r


def _weak(g, n, eps=0.3):
    """exp(eps A): SU(3) links of a smooth field."""
    return _expm(eps * _algebra(g, n))


def _host(t, prec):
    """A tensor of complex numbers as a raw host array."""
    return torch.view_as_real(t.resolve_conj()).reshape(-1).to(torch.float64 if prec == "D" else torch.float32).cpu().numpy()


def _thin(case, g, geo):
    return _weak(g, geo.V * 4).view(geo.V, 4, 3, 3)


def _su3_links(case, g, geo):
    """Forward fat and long links, phases folded in: 1 + 0.3 Gaussian, and SU(3)."""
    fat = 0.3 * _gauss(g, geo.V, 4, 3, 3)
    fat += torch.eye(3, dtype=torch.complex128, device="cuda")
    lng = _weak(g, geo.V * 4).view(geo.V, 4, 3, 3)
    for mu in range(4):
        fat[:, mu] *= geo.sign(mu, 1)[:, None, None]
        lng[:, mu] *= geo.sign(mu, 3)[:, None, None]
    return fat, lng


def _back(geo, fwd, hop):
    return torch.stack([-_dag(fwd[geo.nbr(mu, -hop), mu]) for mu in range(4)], dim=1)


def _rounded(t, prec):
    return t if prec == "D" else t.to(torch.complex64).to(torch.complex128)


def _source(g, geo, n=1):
    """Gaussian source on the even sites."""
    out = []
    for _ in range(n):
        v = _gauss(g, geo.V, 3)
        v[geo.vh:] = 0
        out.append(v)
    return out


def _masses(case):
    sig = np.logspace(np.log10(case["low"]), np.log10(case["low"]) + 3.0, case["nshift"])
    return [float(m) for m in np.sqrt(sig) / 2]


def _terms(case):
    k = np.arange(case["terms"])
    return [float(c) for c in 0.1 * (1.0 + k)]


# ---------------------------------------------------------------- states
_session = None
_live = weakref.WeakSet()


class State:
    """What the caller holds: handles, host arrays, arguments."""

    def __init__(self, case):
        self.case, self.handles = case, []
        _live.add(self)

    def keep(self, h):
        self.handles.append(h)
        return h

    def free(self):
        for h in self.handles:
            h.free()
        self.handles = []

    def __del__(self):
        try:
            self.free()
        except Exception:
            pass


def _open(dims):
    """The session of this lattice (one lattice per process at a time)."""
    global _session
    if _session is None or _session.dims != tuple(dims):
        if _session is not None:
            for st in list(_live):
                st.free()
            _session.close()
        _session = A.Session(dims)
    return _session


def _dims(case):
    return (case["nx"], case["ny"], case["nz"], case["nt"])


def _raw_set(case, g, geo):
    fat, lng = _su3_links(case, g, geo) if case["links"] == "su3" else _smeared(case, _thin(case, g, geo), geo)
    p = case["prec"]
    return [_host(t, p) for t in (fat, lng, _back(geo, fat, 1), _back(geo, lng, 3))]


def _gauge_handle(st, s, case, g, geo):
    return st.keep(A.Gauge(s, _host(_thin(case, g, geo), case["prec"]), prec=case["prec"]))


def _link_handle(st, s, case, g, geo):
    if case["links"] == "su3":
        return st.keep(A.Links(s, *_raw_set(case, g, geo), prec=case["prec"]))
    G = A.Gauge(s, _host(_thin(case, g, geo), case["prec"]), prec=case["prec"])
    L = st.keep(_from_gauge(G, case))
    G.free()
    return L


def _from_gauge(G, case):
    if case["links"] == "hisq":
        return A.LinksFromGauge(G, hisq=True, naik_eps=NAIK_EPS)
    return A.LinksFromGauge(G, coeffs=ASQTAD)


def prepare(case, seed):
    s, geo, g = _open(_dims(case)), Geo(_dims(case)), _gen(seed)
    st, p, kind = State(case), case["prec"], case["kind"]
    st.s = s
    new = lambda n: np.zeros(n, dtype=NP[p])  # noqa: E731
    if kind == "operator":
        st.L = _link_handle(st, s, case, g, geo)
        st.v = [st.keep(A.Vector(s, _host(_gauss(g, geo.V, 3), p), A.EVENODD, p))]
        st.v += [st.keep(A.Vector(s, None, A.EVENODD, p)) for _ in range(2)]
        st.out = new(6 * geo.V)
    elif kind in ("solve", "shifts"):
        st.L = _link_handle(st, s, case, g, geo)
        st.b = _host(_source(g, geo)[0], p)
        st.out = [new(6 * geo.V) for _ in range(case.get("nshift", 1))]
    elif kind == "handover":
        st.raw = _raw_set(case, g, geo)
        st.b = _host(_source(g, geo)[0], p)
        st.out = [new(6 * geo.V)]
    elif kind == "sources":
        st.L = _link_handle(st, s, case, g, geo)
        st.b = [_host(b, p) for b in _source(g, geo, case["nrhs"])]
        st.x = [[st.keep(A.Vector(s, None, A.EVEN, p)) for _ in range(case["nshift"])] for _ in range(case["nrhs"])]
        st.out = [[new(6 * geo.V) for _ in range(case["nshift"])] for _ in range(case["nrhs"])]
    elif kind == "refresh":
        st.G = _gauge_handle(st, s, case, g, geo)
        st.v = [st.keep(A.Vector(s, _host(_gauss(g, geo.V, 3), p), A.EVENODD, p)),
                st.keep(A.Vector(s, None, A.EVENODD, p))]
        st.out = new(6 * geo.V)
    elif kind in ("force", "trajectory"):
        st.U = _host(_thin(case, g, geo), p)
        st.P = _host(_algebra(g, 4 * geo.V), p)
        st.out = [new(72 * geo.V), new(72 * geo.V)]
    elif kind == "outer":
        st.L = _link_handle(st, s, case, g, geo)
        st.x = [st.keep(A.Vector(s, _host(b, p), A.EVEN, p)) for b in _source(g, geo, case["terms"])]
        st.out = [new(72 * geo.V), new(72 * geo.V)]
    else:
        raise ValueError(kind)
    return st


# ---------------------------------------------------------------- one pass
RESID = 1e-20  # squared: a relative residual of 1e-10


def _coeffs():
    return F.symanzik_coeffs(6.0, 0.86)


def _read(st, vec, into):
    st.s.fn(vec.prec, "extract_V_to_raw")(Q.ptr(into), vec.h, vec.parity)
    return into


def _solve(st, L, case):
    b = A.Vector(st.s, st.b, A.EVEN)
    x = A.Vector(st.s, None, A.EVEN)
    if case["method"] == "cg":
        A.invert(L, x, b, case["mass"], A.EVEN, RESID, niter=4000, nrestart=5)
    else:
        A.invert_mixed(L, x, b, case["mass"], A.EVEN, RESID, sloppy_bits=16 if case["method"] == "mixed16" else 32,
                       niter=4000, nrestart=5)
    _read(st, x, st.out[0])
    x.free()
    b.free()
    return st.out


def run(st):
    case = st.case
    kind, p, s = case["kind"], case["prec"], st.s
    if kind == "operator":
        src, a, b = st.v
        for _ in range(case["applications"]):
            A.dslash(st.L, a, src, A.EVEN)
            A.dslash(st.L, a, src, A.ODD)
            src, a, b = a, b, a
        return _read(st, src, st.out)
    if kind == "solve":
        return _solve(st, st.L, case)
    if kind == "handover":
        L = A.Links(s, *st.raw)
        out = _solve(st, L, case)
        L.free()
        return out
    if kind == "shifts":
        m = _masses(case)
        b = A.Vector(s, st.b, A.EVEN)
        x = [A.Vector(s, None, A.EVEN) for _ in m]
        A.invert_multi(st.L, x, b, m, A.EVEN, RESID, niter=4000)
        for v, o in zip(x, st.out):
            _read(st, v, o)
        for v in x + [b]:
            v.free()
        return st.out
    if kind == "sources":
        b = [A.Vector(s, v, A.EVEN) for v in st.b]
        A.invert_multi_rhs(st.L, st.x, b, _masses(case), A.EVEN, RESID, niter=20000, nrestart=2)
        for xs, os_ in zip(st.x, st.out):
            for x, o in zip(xs, os_):
                _read(st, x, o)
        for v in b:
            v.free()
        return st.out
    if kind == "refresh":
        L = _from_gauge(st.G, case)
        A.dslash(L, st.v[1], st.v[0], A.EVEN)
        A.dslash(L, st.v[1], st.v[0], A.ODD)
        _read(st, st.v[1], st.out)
        L.free()
        return st.out
    if kind in ("force", "trajectory"):
        G = A.Gauge(s, st.U, prec=p)
        P = A.Force(s, st.P, prec=p)
        if kind == "force":
            A.gauge_force(G, P, _coeffs(), case["eps"])
        else:
            A.gauge_md(G, P, _coeffs(), case["eps"], case["nsteps"], scheme=1)
            s.fn(p, "extract_G_to_raw")(Q.ptr(st.out[1]), G.h, A.EVENODD)
        s.fn(p, "extract_F_to_raw")(Q.ptr(st.out[0]), P.h, A.EVENODD)
        P.free()
        G.free()
        return st.out[:1] if kind == "force" else st.out
    coef = _terms(case)
    info = Q.Info()
    n = len(coef)
    s.fn(p, "asqtad_fermion_force_oprod")(A.C.byref(info), st.L.h, n, (A.C.c_double * n)(*coef),
                                          (A.C.c_void_p * n)(*[x.h for x in st.x]), Q.ptr(st.out[0]), Q.ptr(st.out[1]))
    return st.out


# ---------------------------------------------------------------- the least work of a pass
def _dslash_work(case, real):
    """Bytes and flops of D onto one parity."""
    vh = int(np.prod(_dims(case))) // 2
    naik = 12 if case["links"] == "su3" else 18
    return vh * (real * (8 * 18 + 8 * naik) + 12 * real), vh * 1146.0


def _steps(case):
    """CG steps to this residual, roughly, as these links and masses need them."""
    m = case["mass"] if "mass" in case else case["low"] ** 0.5 / 2
    return 1000 / (1 + 15 * m) if case["links"] == "su3" else 150 / (1 + 5 * m)


def work(case):
    kind, V = case["kind"], int(np.prod(_dims(case)))
    real = 8 if case["prec"] == "D" else 4
    vh, vec = V // 2, 6 * real * V
    if kind == "operator":
        b, f = _dslash_work(case, real)
        return {"bytes": 2 * case["applications"] * b + vec, "flops": 2 * case["applications"] * f}
    if kind in ("solve", "handover"):
        n = _steps(case)
        b, f = _dslash_work(case, 8 if case["method"] == "cg" else 4)
        v = 9 * (48 if case["method"] == "cg" else 24) * vh
        hand = 4 * 72 * 8 * V if kind == "handover" else 0
        return {"bytes": n * (2 * b + v) + vec + hand, "flops": n * (2 * f + 60 * vh)}
    if kind == "shifts":
        n = _steps(case)
        b, f = _dslash_work(case, 8)
        per = 48 * vh * (7 + 4 * (case["nshift"] - 1) / 8)  # the shifted systems once per 8 steps
        return {"bytes": n * (2 * b + per) + vec * case["nshift"] / 2, "flops": n * (2 * f + 24 * vh * case["nshift"])}
    if kind == "sources":
        n, r = _steps(case), case["nrhs"]
        vec4 = 24 * vh
        link = _dslash_work(case, 4)[0] - 2 * vec4
        per = 2 * link + r * vec4 * (4 + 7 + 4 * (case["nshift"] - 1) / 8)
        return {"bytes": n * per + r * case["nshift"] * vec / 2, "flops": n * r * (2 * 1146.0 + 24 * case["nshift"]) * vh}
    if kind == "refresh":
        # thin links in, fat, long and back links out; staples shared between links: 48
        # products a link for each level
        levels = 2 if case["links"] == "hisq" else 1
        return {"bytes": real * V * (72 + 2 * 144) + 2 * vec,
                "flops": levels * 4.0 * V * 50 * 198}
    if kind in ("force", "trajectory"):
        n = 1 if kind == "force" else 2 * case["nsteps"] + 1
        return {"bytes": real * V * (n * (72 + 2 * 32) + 72 * (3 if kind == "force" else 4)), "flops": n * 4.0 * V * 61.5 * 198}
    n = case["terms"]
    return {"bytes": real * (12 * vh * n + 2 * 72 * V) + _dslash_work(case, real)[0], "flops": n * (4 * V * 2 * 72.0 + 1146.0 * vh)}


# ---------------------------------------------------------------- 64 bits, without the library
def _smeared(case, U, geo):
    """Fat and Naik links of the thin links U with phases, from their path sums."""
    link = lambda mu: U[:, mu]  # noqa: E731

    def staple(W, M, mu, d, s):
        """W_d M W_d^dag displaced by s in direction d, for links along mu."""
        if s > 0:
            return _mm(_mm(W[:, d], M[geo.nbr(d, 1)]), _dag(W[:, d][geo.nbr(mu, 1)]))
        t = _mm(_mm(_dag(W[:, d]), M), W[:, d][geo.nbr(mu, 1)])
        return t[geo.nbr(d, -1)]

    def level(W, c1, c3, c5, c7, cl):
        out = []
        for mu in range(4):
            rest = [d for d in range(4) if d != mu]
            fat = c1 * W[:, mu]
            three = {(f, s): staple(W, W[:, mu], mu, f, s) for f in rest for s in (1, -1)}
            for d in rest:
                e, f = [k for k in rest if k != d]
                inner = c3 * W[:, mu]
                for a, b in ((e, f), (f, e)):
                    m = c5 * W[:, mu] + c7 * (three[b, 1] + three[b, -1])
                    inner = inner + staple(W, m, mu, a, 1) + staple(W, m, mu, a, -1)
                for s in (1, -1):
                    fat = fat + staple(W, inner + cl * three[d, s], mu, d, s)
            out.append(fat)
        return torch.stack(out, dim=1)

    if case["links"] == "hisq":
        X = level(U, 1 / 8, 1 / 16, 1 / 64, 1 / 384, 0.0)
        for _ in range(12):  # polar factor by Newton's iteration
            X = 0.5 * (X + _dag(_inv(X)))
        U = X
        fat = level(U, 1.0, 1 / 16, 1 / 64, 1 / 384, -1 / 8)
        cn = -(1.0 + NAIK_EPS) / 24
    else:
        c1, cn, c3, c5, c7, cl = ASQTAD
        fat = level(U, c1, c3, c5, c7, cl)
    lng = cn * torch.stack([_mm(_mm(link(mu), link(mu)[geo.nbr(mu, 1)]), link(mu)[geo.nbr(mu, 2)]) for mu in range(4)], dim=1)
    for mu in range(4):
        fat[:, mu] *= geo.sign(mu, 1)[:, None, None]
        lng[:, mu] *= geo.sign(mu, 3)[:, None, None]
    return fat, lng


def _inv(a):
    """Inverse of 3x3 matrices by cofactors."""
    rows = [torch.linalg.cross(a[..., (i + 1) % 3, :], a[..., (i + 2) % 3, :]) for i in range(3)]
    det = (a[..., 0, :] * rows[0]).sum(-1)
    return torch.stack(rows, dim=-1) / det[..., None, None]


class Operator:
    """D between the two parities, complex (vh, 3) or (vh, 3, n) vectors."""

    def __init__(self, geo, fat, lng):
        self.t = {0: [], 1: []}
        vh = geo.vh
        for p in (0, 1):
            here, there = slice(p * vh, (p + 1) * vh), (1 - p) * vh
            for mu in range(4):
                for u, hop in ((fat, 1), (lng, 3)):
                    f, b = geo.nbr(mu, hop)[here] - there, geo.nbr(mu, -hop)[here] - there
                    self.t[p].append((u[here, mu], f))
                    self.t[p].append((-_dag(u[b + there, mu]), b))

    def __call__(self, p, v):
        many = v.dim() == 3
        out = torch.zeros_like(v)
        for u, idx in self.t[p]:
            w = v[idx]
            for c in range(3):
                out += u[:, :, c, None] * w[:, c, None, :] if many else u[:, :, c] * w[:, c, None]
        return out


def _exact_links(case, g, geo):
    p = case["prec"]
    if case["links"] == "su3":
        fat, lng = _su3_links(case, g, geo)
        return _rounded(fat, p), _rounded(lng, p)
    return _smeared(case, _rounded(_thin(case, g, geo), p), geo)


def _exact_solve(D, b, masses):
    """(4 m^2 - D D) x = b on the even sites for every mass: multi-shift CG far
    past the library's residual; b is (vh, 3, n)."""
    sig = [4 * m * m for m in masses]
    low = min(range(len(sig)), key=sig.__getitem__)
    dot = lambda u, v: (u.conj() * v).real.sum(dim=(0, 1))  # noqa: E731
    A_ = lambda v: sig[low] * v - D(0, D(1, v))  # noqa: E731
    ds = [s - sig[low] for s in sig]
    n = b.shape[-1]
    x = [torch.zeros_like(b) for _ in sig]
    p = [b.clone() for _ in sig]
    r, rr = b.clone(), dot(b, b)
    stop = 1e-28 * rr
    z0 = [torch.ones(n, device="cuda", dtype=torch.float64) for _ in sig]
    z1 = [z.clone() for z in z0]
    a0, b0 = torch.ones_like(rr), torch.zeros_like(rr)
    for it in range(6000):
        q = A_(p[low])
        a = rr / dot(p[low], q)
        z2 = []
        for j in range(len(sig)):
            z = z1[j] * z0[j] * a0 / (a * b0 * (z0[j] - z1[j]) + z0[j] * a0 * (1 + ds[j] * a))
            z2.append(torch.where(z1[j].abs() > 1e-200, z, torch.zeros_like(z)))
            x[j] = x[j] + p[j] * (a * z2[j] / z1[j].clamp_min(1e-250))
        r = r - q * a
        new = dot(r, r)
        bt = new / rr
        for j in range(len(sig)):
            p[j] = r * z2[j] + p[j] * (bt * (z2[j] / z1[j].clamp_min(1e-250)) ** 2)
        z0, z1, a0, b0, rr = z1, z2, a, bt, new
        if it % 10 == 0 and bool((rr < stop).all()):
            break
    return x


def _full(geo, even):
    out = torch.zeros(geo.V, 3, dtype=torch.complex128, device="cuda")
    out[:geo.vh] = even
    return _host(out, "D")


def _actions(U, geo, c):
    """S = -sum c Re Tr U_loop over plaquettes, rectangles and parallelograms."""
    def step(M, x, mu, s):
        """M followed by the link of direction mu, sense s, from x (an index)."""
        if s > 0:
            return _mm(M, U[x, mu]), geo_n[mu, 1][x]
        y = geo_n[mu, -1][x]
        return _mm(M, _dag(U[y, mu])), y

    geo_n = {(mu, s): geo.nbr(mu, s) for mu in range(4) for s in (1, -1)}
    here = torch.arange(geo.V, device="cuda")

    def loop(path):
        mu, s = path[0]
        M, x = U[here, mu], geo_n[mu, 1]
        for mu, s in path[1:]:
            M, x = step(M, x, mu, s)
        return (M[:, 0, 0] + M[:, 1, 1] + M[:, 2, 2]).real.sum()

    S = 0.0
    for m in range(4):
        for n in range(4):
            if n > m:
                S = S - c[0] * loop([(m, 1), (n, 1), (m, -1), (n, -1)])
            if n != m:
                S = S - c[1] * loop([(m, 1), (m, 1), (n, 1), (m, -1), (m, -1), (n, -1)])
    for a in range(4):
        for b in range(a + 1, 4):
            for d in range(b + 1, 4):
                for s2 in (1, -1):
                    for s3 in (1, -1):
                        S = S - c[2] * loop([(a, 1), (b, s2), (d, s3), (a, -1), (b, -s2), (d, -s3)])
    return S


def _exact_force(U, P, geo, eps):
    """P + eps TA(U g^dag), g the gradient of the action."""
    W = U.clone().requires_grad_(True)
    _actions(W, geo, _coeffs()).backward()
    with torch.no_grad():
        X = _mm(U, _dag(W.grad))
        X = 0.5 * (X - _dag(X))
        tr = (X[..., 0, 0] + X[..., 1, 1] + X[..., 2, 2]) / 3.0
        return P + eps * (X - tr[..., None, None] * torch.eye(3, dtype=torch.complex128, device="cuda"))


def exact(case, seed):
    geo, g, p, kind = Geo(_dims(case)), _gen(seed), case["prec"], case["kind"]
    if kind == "operator":
        D = Operator(geo, *_exact_links(case, g, geo))
        v = _rounded(_gauss(g, geo.V, 3), p)
        for _ in range(case["applications"]):
            v = torch.cat([D(0, v[geo.vh:]), D(1, v[:geo.vh])])
        return _host(v, "D")
    if kind in ("solve", "handover", "shifts"):
        D = Operator(geo, *_exact_links(case, g, geo))
        b = _source(g, geo)[0][:geo.vh]
        m = _masses(case) if kind == "shifts" else [case["mass"]]
        return [_full(geo, x[..., 0]) for x in _exact_solve(D, b[..., None].contiguous(), m)]
    if kind == "sources":
        D = Operator(geo, *_exact_links(case, g, geo))
        b = torch.stack([v[:geo.vh] for v in _source(g, geo, case["nrhs"])], dim=-1)
        xs = _exact_solve(D, b, _masses(case))
        return [[_full(geo, x[..., k]) for x in xs] for k in range(case["nrhs"])]
    if kind == "refresh":
        D = Operator(geo, *_exact_links(case, g, geo))
        v = _rounded(_gauss(g, geo.V, 3), p)
        return _host(torch.cat([D(0, v[geo.vh:]), D(1, v[:geo.vh])]), "D")
    if kind in ("force", "trajectory"):
        U = _rounded(_thin(case, g, geo), p)
        P = _rounded(_algebra(g, 4 * geo.V), p).view(geo.V, 4, 3, 3)
        e = case["eps"] if p == "D" else float(np.float32(case["eps"]))
        if kind == "force":
            return [_host(_exact_force(U, P, geo, e), "D")]
        for k in range(case["nsteps"]):
            P = _exact_force(U, P, geo, (OMELYAN if k == 0 else 2 * OMELYAN) * e)
            U = _mm(_expm(0.5 * e * P), U)
            P = _exact_force(U, P, geo, (1 - 2 * OMELYAN) * e)
            U = _mm(_expm(0.5 * e * P), U)
        P = _exact_force(U, P, geo, OMELYAN * e)
        return [_host(P, "D"), _host(U, "D")]
    D = Operator(geo, *_exact_links(case, g, geo))
    O = [torch.zeros(geo.V, 4, 3, 3, dtype=torch.complex128, device="cuda") for _ in range(2)]
    parity = torch.ones(geo.V, device="cuda", dtype=torch.float64)
    parity[geo.vh:] = -1
    for c, b in zip(_terms(case), _source(g, geo, case["terms"])):
        x = _rounded(b[:geo.vh], p)
        psi = torch.cat([x, D(1, x)])
        for mu in range(4):
            for o, hop in zip(O, (1, 3)):
                o[:, mu] += (c * parity)[:, None, None] * psi[geo.nbr(mu, hop)][:, :, None] * psi.conj()[:, None, :]
    return [_host(o, "D") for o in O]
