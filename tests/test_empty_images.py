"""Empty and negative image sizes are refused with an error code, for the canonical
averaging stencil (whose variant is chosen from the sizes) and for another one.
Runs without a GPU; in a process of its own, which a division by a size of zero
would end."""
import os
import subprocess
import sys

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

CALLS = """
import ctypes, numpy as np
from hindemith_amd import _lib, synthetic as S
L = _lib.lib()
w, ox, oy = S.hs_stencil_taps()["Avg"]
p = lambda a: a.ctypes.data_as(ctypes.c_void_p)
bufs = [np.zeros(64, np.float32) for _ in range(7)]
b = [p(a) for a in bufs]
for nd in (8, 4):  # the first four taps alone are a stencil without a size rule
    for H, W in ((0, 5), (5, 0), (0, 0), (-1, 5), (5, -3)):
        for iters in (0, 7, -1):
            rc = L.hmx_hs_jacobi(b[0], b[1], b[2], None, ctypes.c_float(1.0), H, W, nd, p(w),
                                 p(ox), p(oy), iters, b[3], b[4], b[5], b[6], None)
            assert rc == 1 and b"positive" in L.hmx_last_error(), (nd, H, W, rc)
rc = L.hmx_hs_jacobi(b[0], b[1], b[2], None, ctypes.c_float(1.0), 4, 4, 8, p(w), p(ox), p(oy), -1,
                     b[3], b[4], b[5], b[6], None)
assert rc == 1 and b"iters" in L.hmx_last_error()
print("refused")
"""


def test_jacobi_refuses_empty_images():
    r = subprocess.run([sys.executable, "-c", CALLS], cwd=ROOT, capture_output=True, text=True)
    assert r.returncode == 0 and "refused" in r.stdout, (r.returncode, r.stderr[-500:])
