"""Rounding of the fermion links: their rms distance from the same links in
extended precision is no larger than that of an FP64 evaluation of the same nest
of staples (each product formed by itself, then added), with 10% for the order of
its sums."""
import numpy as np
import pytest

import oracle as O
from conftest import lattice_session
from pyqphix import api as A
from pyqphix import fields as F

DIMS = (8, 8, 8, 8)
# three-link and Lepage terms that nearly cancel, one Naik link
CANCEL = (0, -1 / 24, 1, 1e-3, 0, -1)
HISQ1 = (1 / 8, 0, 1 / 16, 1 / 64, 1 / 384, 0)
HISQ2 = (1, -1 / 24, 1 / 16, 1 / 64, 1 / 384, -1 / 8)


def mul(a, b):
    """a b.  FP64 as the device forms it: an element is one chain of fused
    multiply-adds from zero, each rounded once to 53 bits."""
    if a.dtype != np.complex128:
        return (a[..., :, :, None] * b[..., None, :, :]).sum(-2)
    a, b = a[..., :, :, None], b[..., None, :, :]
    re, im = np.zeros(np.broadcast(a, b).shape[:-3] + (3, 3)), np.zeros(np.broadcast(a, b).shape[:-3] + (3, 3))
    for k in range(3):
        x, y = a[..., :, k, :], b[..., :, k, :]
        for p, q, s in ((x.real, y.real, "re"), (-x.imag, y.imag, "re"), (x.real, y.imag, "im"), (x.imag, y.real, "im")):
            fma = p.astype(np.longdouble) * q + (re if s == "re" else im)
            if s == "re":
                re = fma.astype(np.float64)
            else:
                im = fma.astype(np.float64)
    return re + 1j * im


def smear(lat, U, coef, real):
    """Fat and Naik fields of U[mu][site]; coef as O.ASQTAD."""
    c1, cn, c3, c5, c7, cl = (real(c) for c in coef)
    fwd, bwd = ([lat.shifted(d, h) for d in range(4)] for h in (1, -1))

    def staple(mu, d, s, M):
        if s > 0:
            return mul(mul(U[d], M[fwd[d]]), F.dagger(U[d][fwd[mu]]))
        return mul(mul(F.dagger(U[d][bwd[d]]), M[bwd[d]]), U[d][fwd[mu]][bwd[d]])

    fat, naik = np.empty_like(U), np.empty_like(U)
    for mu in range(4):
        other = [d for d in range(4) if d != mu]
        M = {f: c5 * U[mu] + c7 * staple(mu, f, -1, U[mu]) + c7 * staple(mu, f, 1, U[mu]) for f in other}
        fat[mu] = c1 * U[mu]
        for d in other:
            five = 0
            for e in other:
                if e != d:
                    f = 6 - mu - d - e
                    five = five + staple(mu, e, 1, M[f]) + staple(mu, e, -1, M[f])
            for s in (1, -1):
                N = c3 * U[mu]
                if cl:  # first: its sign is the opposite one
                    N = N + cl * staple(mu, d, s, U[mu])
                fat[mu] = fat[mu] + staple(mu, d, s, N + five)
        u1 = U[mu][fwd[mu]]
        naik[mu] = cn * mul(mul(U[mu], u1), u1[fwd[mu]])
    return fat, naik


def polar(X):
    """Unitary polar factor: Newton iterations, the inverse by cofactors."""
    for _ in range(12):
        A3 = np.empty_like(X)
        for i in range(3):
            for j in range(3):
                i1, i2, j1, j2 = (i + 1) % 3, (i + 2) % 3, (j + 1) % 3, (j + 2) % 3
                A3[..., j, i] = X[..., i1, j1] * X[..., i2, j2] - X[..., i1, j2] * X[..., i2, j1]
        det = (X[..., 0, :] * A3[..., :, 0]).sum(-1)
        inv = A3 * (det.conj() / (det.real ** 2 + det.imag ** 2))[..., None, None]
        X = X.real.dtype.type(0.5) * (X + F.dagger(inv))
    return X


def links(lat, U, coef, real, cplx):
    """Of asqtad coefficients, or HISQ with None."""
    u = np.moveaxis(U, 1, 0).astype(cplx)
    if coef is None:
        u = polar(smear(lat, u, HISQ1, real)[0])
    out = []
    for a, hop in zip(smear(lat, u, coef or HISQ2, real), (1, 3)):
        a = np.moveaxis(a, 0, 1).copy()
        for mu in range(4):
            a[:, mu] *= (lat.eta(mu) * lat.bc(mu, hop))[:, None, None]
        out.append(a)
    return out


def rms(a, ref):
    return float(np.sqrt((np.abs(a.astype(ref.dtype) - ref) ** 2).mean() / (np.abs(ref) ** 2).mean()))


@pytest.mark.gpu
@pytest.mark.parametrize("seed,eps", [(31, 0.5), (33, 0.15)])  # rough, and smooth
@pytest.mark.parametrize("kind", ["asqtad", "cancelling", "hisq"])
def test_links_as_close_to_extended_precision_as_fp64_allows(kind, seed, eps):
    s, lat = lattice_session(DIMS), F.Lattice(DIMS)
    U = F.gauge_field(lat, "weak", seed, eps=eps)
    coef = {"asqtad": O.ASQTAD, "cancelling": CANCEL, "hisq": None}[kind]
    print(f"[case] link accuracy {kind} eps {eps}", flush=True)
    G = A.Gauge(s, F.to_raw(U))
    L = A.LinksFromGauge(G, coeffs=coef) if coef else A.LinksFromGauge(G, hisq=True)
    got = [F.from_raw_links(a, lat) for a in L.extract()]
    exact = links(lat, U, coef, np.longdouble, np.clongdouble)
    fp64 = links(lat, U, coef, np.float64, np.complex128)
    for g, f, e in zip(got, fp64, exact):
        assert f.dtype == np.complex128 and np.finfo(e.real.dtype).nmant >= 63
        assert rms(g, e) < 1.1 * rms(f, e)
    for o in (L, G):
        o.free()
