"""The Dslash's launch shapes at their edges: four lanes per site in blocks of 64
and of 256 work-items, one lane per site with cached links, and with streamed
ones (by the link type), each with every epilogue.  The plain operator against
the oracle (FP64 1e-13, FP32 1e-6 relative); the solvers' reductions through the
residual that the oracle's operator finds in their solutions."""
import numpy as np
import pytest

import oracle as O
from conftest import lattice_session
from helpers import half, rel_l2
from pyqphix import api as A
from pyqphix import fields as F

pytestmark = pytest.mark.gpu
NP = {"D": np.float64, "F": np.float32}
# sites per parity: 128; 2688 (168 blocks of 16); 19200 and 20480, either side of
# the small blocks; 38400 and 40960, either side of four lanes; 76800 (FP64 links
# streamed, FP32 ones cached)
DIMS = [(4, 4, 4, 4), (4, 12, 28, 4), (8, 12, 20, 20), (8, 16, 16, 20), (12, 16, 20, 20), (16, 16, 16, 20),
        (12, 20, 20, 32)]


@pytest.mark.parametrize("kind", ["haar", "scaled"])
@pytest.mark.parametrize("dims", DIMS)
def test_operator_and_solvers(dims, kind):
    s = lattice_session(dims)
    lat = F.Lattice(dims)
    fat, lng = F.make_links(lat, "haar", 21)
    if kind == "scaled":  # 18-real Naik links
        lng = lng * (-1.0 / 24)
    raw = F.raw_link_set(lat, fat, lng)
    orc = O.Oracle(dims, *raw)
    psi = F.to_raw(F.gaussian_source(lat, 22))
    print(f"[case] shapes {dims} {kind}", flush=True)
    for prec, tol in (("D", 1e-13), ("F", 1e-6)):
        L = A.Links(s, *[r.astype(NP[prec]) for r in raw], prec=prec)
        vin = A.Vector(s, psi.astype(NP[prec]), A.EVENODD, prec)
        out = A.Vector(s, None, A.EVENODD, prec)
        A.dslash(L, out, vin, A.EVEN)
        A.dslash(L, out, vin, A.ODD)
        got = out.extract()
        for cb in (0, 1):
            assert rel_l2(half(got, lat, cb), orc.dslash(half(psi, lat, 1 - cb), cb)) < tol
        for o in (L, vin, out):
            o.free()
    L = A.Links(s, *raw)
    mass = 0.3
    b = F.to_raw(F.gaussian_source(lat, 23, parity=0))
    vb, vx = A.Vector(s, b, A.EVEN), A.Vector(s, None, A.EVEN)
    hb = half(b, lat, 0)

    def residual():
        x = half(vx.extract(), lat, 0)
        r = hb - 4 * mass * mass * x + orc.dslash(orc.dslash(x, 1), 0)
        return np.linalg.norm(r) / np.linalg.norm(hb)

    def solve(fn, **kw):
        nonlocal vx
        vx.free()
        vx = A.Vector(s, None, A.EVEN)
        ret, info, res = fn(L, vx, vb, mass, A.EVEN, 1e-18, niter=2000, **kw)
        assert info.status == 0 and residual() < 1.01e-9

    try:
        for fs in (2, 3):  # the plain CG's two-reduction and single-reduction steps
            s.lib.QPHIX_MI355X_set_fewsums(fs)
            solve(A.invert)
        for bits in (32, 16):
            for link_bits in (32, 16):
                s.lib.QPHIX_MI355X_set_sloppy_link_bits(link_bits)
                for fs in (2, 0):
                    s.lib.QPHIX_MI355X_set_fewsums(fs)
                    solve(A.invert_mixed, sloppy_bits=bits)
    finally:
        s.lib.QPHIX_MI355X_set_fewsums(2)
        s.lib.QPHIX_MI355X_set_sloppy_link_bits(32)
    for o in (L, vb, vx):
        o.free()
