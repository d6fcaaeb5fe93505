"""What hs_tune measured is used for the stencil and the solves that it measured."""
import numpy as np
import pytest
import torch

import oracle
from hindemith_amd import kernels as K
from hindemith_amd import synthetic as S

pytestmark = pytest.mark.gpu
TAPS = S.hs_stencil_taps()
AVG9 = (np.full(9, 1.0 / 9.0, np.float32), np.array([-1, 0, 1] * 3, np.int32),
        np.repeat(np.array([-1, 0, 1], np.int32), 3))


def test_tuning_another_stencil_leaves_the_canonical_choice():
    H, W = 101, 163
    planes = [torch.randn(H, W, device="cuda") * 0.1 for _ in range(3)]
    before = K.hs_config(H, W)
    vi, k = K.hs_tune(*planes, 1.0, AVG9)
    # the row-register variants have no kernel of their own for this stencil
    assert K.hs_variants()[vi]["kernel"] != "hs_rows_kernel" and 1 <= k <= 8
    assert K.hs_config(H, W) == before
    chosen = K.hs_tune(*planes, 1.0, TAPS["Avg"])
    assert K.hs_config(H, W) == chosen
    # solves of both stencils, short and long, after both
    I1, I2, _, _ = S.hs_pair(H, W, seed=3)
    d1, d2 = torch.from_numpy(I1).cuda(), torch.from_numpy(I2).cuda()
    for avg in (TAPS["Avg"], AVG9):
        taps = dict(TAPS, Avg=avg)
        for iters in (7, 101):
            u, v = K.hs_solve(d1, d2, 1.0, taps, iters)
            ru, rv = oracle.hs_solve(I1, I2, 1.0, taps, iters)
            assert np.array_equal(u.cpu().numpy(), ru) and np.array_equal(v.cpu().numpy(), rv)
