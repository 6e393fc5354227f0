"""The plain CG where its vector kernels have more blocks than the card holds at
once (32^3 x 64: 2048 of 512 work-items, against 768 in FP64 and at most 1024 in
FP32): blocks that start after the step's stopping rule was met update x as well.
The same steps with a relative residue that any solution meets take x in the
kernel before and are the reference: the same arithmetic in the same order, so
x agrees to rounding (a block without its last update is off by 1e-3 or more of
the largest element)."""
import numpy as np
import pytest

import oracle as O
from conftest import lattice_session
from helpers import half, rel_l2
from pyqphix import api as A
from pyqphix import fields as F

pytestmark = pytest.mark.gpu
NP = {"D": np.float64, "F": np.float32}
SMALL, BIG = (8, 8, 8, 8), (32, 32, 32, 64)


def repeated(ls, lb, raw):
    """A small lattice's raw array repeated over the big one."""
    at = ls.index(lb.x, lb.y, lb.z, lb.t)
    return np.ascontiguousarray(raw.reshape(ls.V, -1)[at]).ravel()


@pytest.mark.parametrize("prec,tol", [("D", 1e-12), ("F", 1e-5)])
def test_every_block_takes_the_last_update(prec, tol):
    s = lattice_session(BIG)
    ls, lb = F.Lattice(SMALL), F.Lattice(BIG)
    fat, lng = F.make_links(ls, "weak", 61)
    L = A.Links(s, *[repeated(ls, lb, r.astype(NP[prec])) for r in F.raw_link_set(ls, fat, lng)], prec=prec)
    b = np.random.default_rng(62).standard_normal(6 * lb.V).astype(NP[prec])
    vb = A.Vector(s, b, A.EVEN, prec)
    # one inner loop that ends at its limit; restarts at every limit until converged
    for niter, nrestart, resid in ((7, 1, 1e-30), (12, 40, 1e-9 if prec == "F" else 1e-18)):
        got = []
        for relresid in (0.0, 1e30):
            print(f"[case] CG blocks {prec} niter {niter} relresid {relresid}", flush=True)
            vx = A.Vector(s, None, A.EVEN, prec)
            _, info, res = A.invert(L, vx, vb, 0.3, A.EVEN, resid, relresid=relresid, niter=niter, nrestart=nrestart)
            assert info.status == 0
            got.append((vx.extract(), res.final_iter, res.final_restart, res.final_rsq))
            vx.free()
        (x, it, rs, rsq), (y, ity, rsy, rsqy) = got
        assert (it, rs) == (ity, rsy)
        assert np.abs(x - y).max() < tol * np.abs(y).max()
        assert abs(rsq - rsqy) < max(tol, 1e-6) * rsqy
        if nrestart > 1:
            assert rsq < resid
    for o in (L, vb):
        o.free()


@pytest.mark.parametrize("dims", [(24, 32, 32, 32), (32, 32, 32, 32)])  # 393216 and 524288 sites per parity
def test_operator_either_side_of_the_small_blocks(dims):
    """Streamed links in blocks of 64 work-items and of 256 (400000 sites): on a
    repeated small lattice the operator repeats that lattice's, which the oracle
    gives (FP64 1e-13, FP32 1e-6 relative)."""
    s = lattice_session(dims)
    ls, lb = F.Lattice(SMALL), F.Lattice(dims)
    raw = F.raw_link_set(ls, *F.make_links(ls, "weak", 63))
    orc = O.Oracle(SMALL, *raw)
    psi = F.to_raw(F.gaussian_source(ls, 64))
    want = np.concatenate([orc.dslash(half(psi, ls, 1 - cb), cb) for cb in (0, 1)])
    for prec, tol in (("D", 1e-13), ("F", 1e-6)):
        print(f"[case] operator {dims} {prec}", flush=True)
        L = A.Links(s, *[repeated(ls, lb, r.astype(NP[prec])) for r in raw], prec=prec)
        vin = A.Vector(s, repeated(ls, lb, psi.astype(NP[prec])), A.EVENODD, prec)
        out = A.Vector(s, None, A.EVENODD, prec)
        A.dslash(L, out, vin, A.EVEN)
        A.dslash(L, out, vin, A.ODD)
        assert rel_l2(out.extract(), repeated(ls, lb, want)) < tol
        for o in (L, vin, out):
            o.free()
