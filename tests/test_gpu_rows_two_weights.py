"""Row-register sweeps with two averaging weights (the builds that hold them in two
registers), and with weights that differ from two in one place, which take the
eight-weight builds: every variant at window edges, bit for bit against the oracle."""
import numpy as np
import pytest
import torch

import oracle
from hindemith_amd import kernels as K
from hindemith_amd import synthetic as S

pytestmark = pytest.mark.gpu
TAPS = S.hs_stencil_taps()
TWO = np.array([0.17] * 4 + [0.08] * 4, np.float32)


@pytest.mark.parametrize("changed", [None, 1, 3, 5, 7])
@pytest.mark.parametrize("shape", [(1, 64), (17, 47), (33, 63), (65, 130), (150, 62)])
def test_two_weight_builds_bitexact(shape, changed):
    w = TWO.copy()
    if changed is not None:
        w[changed] = np.nextafter(w[changed], np.float32(1))
    avg = (w, TAPS["Avg"][1], TAPS["Avg"][2])
    rng = np.random.default_rng(shape[0] * 7 + shape[1])
    mk = lambda s: (s * rng.normal(size=shape)).astype(np.float32)  # noqa: E731
    Ix, Iy, It, u0, v0 = mk(0.3), mk(0.3), mk(0.1), mk(1.0), mk(1.0)
    dev = lambda a: torch.from_numpy(a).cuda()  # noqa: E731
    ref = oracle.hs_jacobi(Ix, Iy, It, 0.7, avg, 17, u0, v0)
    dIx, dIy, dIt = dev(Ix), dev(Iy), dev(It)
    for vi, v in enumerate(K.hs_variants()):
        if v["kernel"] != "hs_rows_kernel":
            continue
        for k in (1, 2, 8, v["kmax"]):
            u, vv = dev(u0), dev(v0)
            K.hs_jacobi(dIx, dIy, dIt, 0.7, avg, 17, u, vv, variant=vi, k=k)
            assert np.array_equal(u.cpu().numpy(), ref[0]), (vi, k)
            assert np.array_equal(vv.cpu().numpy(), ref[1]), (vi, k)
