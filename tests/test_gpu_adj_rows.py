"""The adjoint's fused reverse blocks (hs_adj_rows.h) against the two-launch form.

Both perform the same arithmetic in the same order, so the gradients are equal;
the two-launch form is pinned by the fp64 oracle and finite differences
(test_gpu_adjoint.py).  Sizes at the edges of windows and strips, one row or
column, every block length, and batches large enough for each build."""
import numpy as np
import pytest
import torch

from hindemith_amd.autograd import horn_schunck
from hindemith_amd import synthetic as S

pytestmark = pytest.mark.gpu
TAPS = S.hs_stencil_taps()
AVG = (np.array([0.11, 0.17, 0.13, 0.19, 0.07, 0.12, 0.05, 0.16], np.float32),) + \
    tuple(TAPS["Avg"][1:])


def _grads(shape, iters, every, start, seed, taps):
    g = torch.Generator(device="cuda").manual_seed(seed)
    rnd = lambda *s: torch.randn(*s, generator=g, device="cuda")  # noqa: E731
    B = shape[0]
    wrt = [rnd(*shape), rnd(*shape), 0.5 + torch.rand(B, generator=g, device="cuda")]
    if start:
        wrt += [rnd(*shape), rnd(*shape)]
    for t in wrt:
        t.requires_grad_(True)
    u0, v0 = (wrt[3], wrt[4]) if start else (None, None)
    u, v = horn_schunck(*wrt[:3], iters=iters, ckpt_every=every, taps=taps, u0=u0, v0=v0)
    return [u.detach(), v.detach()] + list(torch.autograd.grad([u, v], wrt,
                                                               [rnd(*shape), rnd(*shape)]))


@pytest.mark.parametrize("shape,iters,every,start", [
    ((1, 1, 1), 3, 3, False), ((1, 2, 3), 5, 2, True), ((2, 1, 70), 9, 4, True),
    ((2, 70, 1), 9, 8, False), ((1, 16, 48), 1, 1, True), ((1, 17, 49), 2, 2, True),
    ((1, 33, 65), 8, 8, True), ((2, 31, 50), 17, 20, True), ((1, 47, 97), 23, 9, False),
    ((1, 64, 129), 300, 12, False), ((3, 150, 62), 14, 7, True), ((3, 243, 331), 21, 5, True),
    ((2, 512, 512), 24, 8, True), ((7, 301, 403), 11, 6, False)])
def test_fused_blocks_match_two_launch_form(shape, iters, every, start, monkeypatch):
    taps = dict(TAPS, Avg=AVG)
    got = _grads(shape, iters, every, start, 3, taps)
    monkeypatch.setenv("HMX_ADJ_GENERIC", "1")
    ref = _grads(shape, iters, every, start, 3, taps)
    for a, b in zip(got, ref):
        assert torch.equal(a, b)
