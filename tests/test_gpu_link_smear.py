"""The staged smearing passes at the edges of their launch shapes.

Small lattices against the oracle's path-by-path links: fewer sites than one
block of 256, a partly empty block, whole blocks walked by z-region.  A lattice
whose scratch is over the kept workspace takes one direction at a time; its thin
field repeats a small lattice's, so its links must repeat that lattice's links
bit for bit (the same sums in the same order)."""
import numpy as np
import pytest

import oracle as O
from conftest import lattice_session
from helpers import rel_l2
from pyqphix import api as A
from pyqphix import fields as F

pytestmark = pytest.mark.gpu


def build(s, U, kind, prec="D", periodic=False):
    G = A.Gauge(s, U, prec=prec)
    if kind == "hisq":
        L = A.LinksFromGauge(G, hisq=True, naik_eps=0.05, periodic_t=periodic)
    else:
        L = A.LinksFromGauge(G, coeffs=O.ASQTAD, periodic_t=periodic)
    out = L.extract()
    L.free()
    G.free()
    return out


@pytest.mark.parametrize("kind", ["asqtad", "hisq"])
@pytest.mark.parametrize("dims", [(4, 4, 4, 4), (12, 4, 4, 4), (4, 12, 8, 4), (8, 8, 8, 16)])
def test_smeared_links_by_launch_shape(dims, kind):
    s = lattice_session(dims)
    lat = F.Lattice(dims)
    U = F.to_raw(F.gauge_field(lat, "weak", 31, eps=0.5))
    print(f"[case] smear {dims} {kind}", flush=True)
    fat, lng = build(s, U, kind)
    if kind == "hisq":
        fo, lo = O.links_from_gauge(dims, U, hisq=True, naik_eps=0.05)
    else:
        fo, lo = O.links_from_gauge(dims, U, coef=O.ASQTAD)
    # ~170 products of FP64 rounding 1e-16 per link: well inside 1e-13
    assert rel_l2(fat, fo) < 1e-13 and rel_l2(lng, lo) < 1e-13


def test_one_direction_at_a_time_repeats_the_small_lattice():
    small, big = (8, 8, 4, 4), (32, 32, 32, 20)
    ls, lb = F.Lattice(small), F.Lattice(big)
    U = F.gauge_field(ls, "weak", 32, eps=0.5)
    print(f"[case] smear {big} repeating {small}", flush=True)
    fat, lng = build(lattice_session(small), F.to_raw(U), "hisq", periodic=True)
    at = ls.index(lb.x, lb.y, lb.z, lb.t)
    rep = lambda a: np.ascontiguousarray(a.reshape(ls.V, 72)[at]).ravel()
    fb, lngb = build(lattice_session(big), rep(F.to_raw(U)), "hisq", periodic=True)
    assert np.array_equal(fb, rep(fat)) and np.array_equal(lngb, rep(lng))
