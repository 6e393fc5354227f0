"""Chunked transfers between raw host arrays and the device: every field comes
back as it was given, over one chunk and many, part of a last chunk, one parity
and both, pageable, pinned and device memory, and several threads at once; the
long links' storage is decided the same wherever the first link that is not
SU(3) lies."""
import ctypes as C
import threading

import numpy as np
import pytest
import torch

from conftest import lattice_session
from helpers import random_links
from pyqphix import api as A
from pyqphix import fields as F

pytestmark = pytest.mark.gpu
NP = {"D": np.float64, "F": np.float32}
# 0.2 MB vectors (the kernels use the pinned buffers), then several chunks, then
# chunks that do not divide a parity
DIMS = [(4, 4, 4, 8), (8, 8, 8, 8), (16, 16, 16, 16), (20, 12, 16, 28)]


def momenta(rng, V, dt):
    a = F.antihermitian_traceless(rng, (V, 4)).astype(np.complex128 if dt == np.float64 else np.complex64)
    for k in range(3):
        a[..., k, k] = 1j * a[..., k, k].imag
    a[..., 2, 2] = -1j * (a[..., 0, 0].imag + a[..., 1, 1].imag)
    for r, c in ((1, 0), (2, 0), (2, 1)):
        a[..., r, c] = -np.conj(a[..., c, r])
    return np.ascontiguousarray(a).view(dt).ravel()


@pytest.mark.parametrize("prec", ["D", "F"])
@pytest.mark.parametrize("dims", DIMS)
def test_fields_round_trip(dims, prec):
    s = lattice_session(dims)
    V = s.V
    print(f"[case] round trip {dims} {prec}", flush=True)
    rng = np.random.default_rng(3)
    v = rng.standard_normal(6 * V).astype(NP[prec])
    for parity in (A.EVEN, A.ODD, A.EVENODD):
        x = A.Vector(s, v, parity, prec)
        got, want = x.extract(), np.zeros_like(v)
        for p, bit in ((0, A.EVEN), (1, A.ODD)):
            if parity & bit:
                want[3 * p * V:3 * (p + 1) * V] = v[3 * p * V:3 * (p + 1) * V]
        assert np.array_equal(got, want)
        x.free()
    u = rng.standard_normal(72 * V).astype(NP[prec])
    m = momenta(rng, V, NP[prec])
    for cls, raw in ((A.Gauge, u), (A.Force, m)):
        x = cls(s, raw, prec=prec)
        assert np.array_equal(x.extract(), raw)
        one = x.extract(A.ODD)
        assert not one[:36 * V].any() and np.array_equal(one[36 * V:], raw[36 * V:])
        x.free()


@pytest.mark.parametrize("where", ["none", "first", "last"])
@pytest.mark.parametrize("dims", DIMS[1:])
def test_long_link_storage_wherever_it_is_decided(dims, where):
    s = lattice_session(dims)
    lat = F.Lattice(dims)
    print(f"[case] long links {dims} {where}", flush=True)
    raw = [F.to_raw(a) for a in random_links(lat, "haar", 4)]
    if where != "none":  # one element of one long link off SU(3): forward at the first site, back at the last
        raw[1 if where == "first" else 3][12 if where == "first" else -6] += 0.25
    L = A.Links(s, *raw)
    assert L.recon == (12 if where == "none" else 18)
    s.lib.QPHIX_MI355X_set_long_recon(18)
    try:
        L18 = A.Links(s, *raw)
    finally:
        s.lib.QPHIX_MI355X_set_long_recon(0)
    fat, lng = L.extract()
    assert np.array_equal(fat, raw[0])
    assert np.abs(lng - raw[1]).max() < (1e-14 if where == "none" else 1e-300)
    vin = A.Vector(s, F.to_raw(F.gaussian_source(lat, 5)), A.EVENODD)
    a, b = A.Vector(s, None, A.EVENODD), A.Vector(s, None, A.EVENODD)
    for p in (A.EVEN, A.ODD):
        A.dslash(L, a, vin, p)
        A.dslash(L18, b, vin, p)
    x, y = a.extract(), b.extract()
    assert np.array_equal(x, y) if where != "none" else np.linalg.norm(x - y) < 1e-14 * np.linalg.norm(y)
    for o in (L, L18, vin, a, b):
        o.free()


def test_pinned_and_device_arrays():
    s = lattice_session((16, 16, 16, 16))
    print("[case] pinned and device raw arrays", flush=True)
    want = torch.randn(6 * s.V, dtype=torch.float64)
    pinned = torch.empty(6 * s.V, dtype=torch.float64, pin_memory=True).copy_(want)
    dev = want.cuda()
    torch.cuda.synchronize()
    for src in (pinned, dev):
        h = s.fn("D", "create_V_from_raw")(C.c_void_p(src.data_ptr()), A.EVENODD)
        out = torch.zeros_like(src)
        torch.cuda.synchronize()
        s.fn("D", "extract_V_to_raw")(C.c_void_p(out.data_ptr()), h, A.EVENODD)
        assert torch.equal(out.cpu(), want)
        s.fn("D", "destroy_V")(h)


def test_several_threads():
    s = lattice_session((16, 16, 16, 16))
    print("[case] transfers from four threads", flush=True)
    bad = []

    def work(k):
        raw = np.random.default_rng(k).standard_normal(6 * s.V)
        for _ in range(10):
            v = A.Vector(s, raw, A.EVENODD)
            if not np.array_equal(v.extract(), raw):
                bad.append(k)
            v.free()

    th = [threading.Thread(target=work, args=(k,)) for k in range(4)]
    [t.start() for t in th]
    [t.join() for t in th]
    assert not bad
