"""Device memory that the link preparation used is there for others: with the card
nearly full, fields fit that need it back."""
import numpy as np
import pytest
import torch

from conftest import lattice_session
from pyqphix import api as A
from pyqphix import fields as F

pytestmark = pytest.mark.gpu


def test_link_preparation_gives_its_scratch_back():
    dims = (24, 24, 20, 28)  # of no other test: nothing is held yet
    s = lattice_session(dims)
    lat = F.Lattice(dims)
    one = np.zeros((lat.V, 4, 3, 3), dtype=np.complex128)
    one[...] = np.eye(3)
    U = F.to_raw(one)
    G = A.Gauge(s, U)
    before = torch.cuda.mem_get_info()[0]
    A.LinksFromGauge(G, hisq=True).free()
    held = before - torch.cuda.mem_get_info()[0]
    print(f"[case] scratch: {held / 2**30:.2f} GiB held after a link preparation", flush=True)
    left = 2 << 30
    fill = torch.empty(torch.cuda.mem_get_info()[0] - left, dtype=torch.uint8, device="cuda")
    fields = []
    s.lib.QPHIX_MI355X_set_abort_on_error(0)  # no memory: a test that fails, not an exit
    try:
        per = 8 * 72 * s.V * 5 // 3  # links and their two-row copy
        n = (left + held * 3 // 4) // per
        assert n * per > left + (1 << 30)  # more than is free: the rest is the scratch's
        for _ in range(n):
            fields.append(A.Gauge(s, U))
            assert fields[-1].h
        assert np.array_equal(fields[-1].extract(), U)
    finally:
        s.lib.QPHIX_MI355X_set_abort_on_error(1)
        for g in fields + [G]:
            g.free()
        del fill
        torch.cuda.empty_cache()
