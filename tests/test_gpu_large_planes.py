"""Images whose planes pass 4 GiB: every kernel's row addresses are 64 bits.

A pixel depends on the rows within a few of its own, so the last rows of a large
image equal those of its last rows taken as an image, bit for bit (all operations
are the same; the crop's own upper rows differ, as far as the iterations reach).
The image's last 126 rows lie past the 32-bit byte offsets."""
import ctypes

import numpy as np
import pytest
import torch

from hindemith_amd import autograd as AG
from hindemith_amd import kernels as K
from hindemith_amd import synthetic as S
from hindemith_amd._lib import check, lib

pytestmark = pytest.mark.gpu
TAPS = S.hs_stencil_taps()
AVG5 = (np.full(5, 0.2, np.float32), np.int32([0, -1, 1, 0, 0]), np.int32([0, 0, 0, -1, 1]))
H, W, CROP, LAST = 32640, 33024, 160, 120


def _need(planes):
    torch.cuda.empty_cache()
    if torch.cuda.mem_get_info()[0] < planes * H * W * 4 + (4 << 30):
        pytest.skip("not enough free device memory")


def _plane(seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    return torch.randn(H, W, generator=g, device="cuda")


@pytest.mark.parametrize("avg", [TAPS["Avg"], AVG5], ids=["canonical", "five"])
@pytest.mark.parametrize("iters", [1, 9])
def test_solve_past_4gib(avg, iters):
    _need(11)
    taps = dict(TAPS, Avg=avg)
    I1, I2 = _plane(1), _plane(2)
    u, v = K.hs_solve(I1, I2, 1.0, taps, iters)
    cu, cv = K.hs_solve(I1[-CROP:].clone(), I2[-CROP:].clone(), 1.0, taps, iters)
    assert torch.equal(u[-LAST:], cu[-LAST:]) and torch.equal(v[-LAST:], cv[-LAST:])
    fu, fv = K.hs_solve(I1[:CROP].clone(), I2[:CROP].clone(), 1.0, taps, iters)
    assert torch.equal(u[:LAST], fu[:LAST]) and torch.equal(v[:LAST], fv[:LAST])


def _adjoint(I1, I2, ck, gu, taps):
    """Gradients of the frames from one step's adjoint, through the C ABI."""
    h = I1.shape[0]
    L, null = lib(), ctypes.c_void_p(0)
    keep, targs = AG._tap_args(taps)
    al = torch.ones(1, device="cuda")
    g1, g2, ga = torch.empty_like(I1), torch.empty_like(I1), torch.empty(1, device="cuda")
    ws = torch.empty(int(L.hmx_hs_adjoint_workspace(1, h, W, 1)) // 4 + 1, device="cuda")
    check(L.hmx_hs_adjoint(K._ptr(I1), K._ptr(I2), 1, h, W, K._ptr(al), *targs, 1, 1, K._ptr(ck),
                           null, null, K._ptr(gu), K._ptr(gu), K._ptr(g1), K._ptr(g2), K._ptr(ga),
                           null, null, K._ptr(ws), K.stream_ptr()), "adjoint")
    torch.cuda.synchronize()
    return g1, g2


def test_adjoint_past_4gib():
    _need(27)
    I1, I2, gu = _plane(1), _plane(2), _plane(3)
    ck = torch.empty(2, H, W, device="cuda")
    ck[0], ck[1] = _plane(4), _plane(5)
    g1, g2 = _adjoint(I1, I2, ck, gu, TAPS)
    crop = lambda t: t[..., -CROP:, :].clone()  # noqa: E731
    c1, c2 = _adjoint(crop(I1), crop(I2), crop(ck), crop(gu), TAPS)
    assert torch.equal(g1[-LAST:], c1[-LAST:]) and torch.equal(g2[-LAST:], c2[-LAST:])
