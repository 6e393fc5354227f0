"""An error that ends the process in the middle of a transfer (out of memory while
the long links are stored anew, with abort_on_error set) still ends it when an exit
handler finalizes the library."""
import os
import subprocess
import sys

import pytest

pytestmark = pytest.mark.gpu
ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
PROGRAM = """
import ctypes as C, sys
sys.path[:0] = [{root!r} + "/milc-qphix_amd"]
import numpy as np
from pyqphix import api as A
s = A.Session((16, 16, 16, 16))
raw = np.random.default_rng(1).standard_normal(72 * s.V)  # not SU(3): 18 reals, decided in the first chunk
A.Links(s, raw, raw, raw, raw).free()
C.CDLL(None).__cxa_atexit(C.cast(s.lib.QPHIX_finalize, C.c_void_p), None, None)
s.lib.QPHIX_MI355X_set_abort_on_error(1)
# staging, maximum, two fat parities, two signs and two long ones; then the new long ones
s.lib.QPHIX_MI355X_debug_fail_alloc(8)
print("[case] exit inside a transfer", flush=True)
A.Links(s, raw, raw, raw, raw)
"""


def test_exit_inside_a_transfer():
    r = subprocess.run([sys.executable, "-u", "-c", PROGRAM.format(root=ROOT)], capture_output=True, text=True, timeout=100)
    assert "[case] exit inside a transfer" in r.stdout, r.stderr
    assert r.returncode == 1 and "QPHIX ERROR" in r.stderr and "[injected]" in r.stderr, (r.returncode, r.stderr)
