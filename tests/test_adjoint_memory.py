"""What the adjoint allocates (no GPU involved): the canonical stencil's fused blocks keep
the state before each 8-step block but a segment's first, any other stencil two planes per
step; and autograd's checkpoints with them stay within the bound that it states."""
import numpy as np
import pytest

from hindemith_amd import autograd as AG
from hindemith_amd import synthetic as S
from hindemith_amd._lib import lib
from hindemith_amd.kernels import _Taps

AVG = S.hs_stencil_taps()["Avg"]
AVG5 = (np.full(5, 0.2, np.float32), np.int32([0, -1, 1, 0, 0]), np.int32([0, 0, 0, -1, 1]))
B, H, W = 2, 30, 40
PAIR = 2 * B * H * W * 4
FIXED = 11 * B * H * W * 4 + B * 4 + 256 + B * 64 * 8  # planes and words of every form


def _pairs(every, avg):
    t = _Taps(avg)
    extra = lib().hmx_hs_adjoint_workspace_taps(B, H, W, every, *t.args()) - FIXED
    assert extra >= 0 and extra % PAIR == 0
    return extra // PAIR


@pytest.mark.parametrize("every,fused", [(1, 0), (8, 0), (9, 2), (16, 2), (17, 3), (50, 7)])
def test_workspace_by_stencil(every, fused, monkeypatch):
    assert _pairs(every, AVG) == fused
    assert _pairs(every, AVG5) == every + 2
    assert lib().hmx_hs_adjoint_workspace(B, H, W, every) == FIXED + PAIR * (every + 2)
    for switch in ("HMX_ADJ_GENERIC", "HMX_LIN_STAGED"):  # the two-launch form
        monkeypatch.setenv(switch, "1")
        assert _pairs(every, AVG) == every + 2
        monkeypatch.delenv(switch)


def test_bad_stencil_is_refused():
    t = _Taps(AVG)
    assert lib().hmx_hs_adjoint_workspace_taps(B, H, W, 8, 0, *t.args()[1:]) < 0


def test_stated_bound_holds():
    for iters in list(range(1, 70)) + [100, 200, 201, 500, 1000]:
        for every in (1, 2, 3, 7, 8, 9, 12, 16, 20, 32, 50):
            seg = AG._segment(iters, every)
            pairs = -(-iters // seg) + _pairs(seg, AVG)
            assert pairs <= -(-iters // every) + every, (iters, every, seg, pairs)
