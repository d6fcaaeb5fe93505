"""The adjoint with averaging stencils other than the canonical one (the two-launch form:
a recompute that stores each step's linearisation, and hs_adj_tb_kernel), the
linearisation that the forward keeps for it, and the checkpoint intervals of both forms
through the C ABI (autograd picks the canonical stencil's interval itself).

Against the fp64 reverse-mode oracle: 1e-3 of the gradient's norm, float32's error over
these step counts with room, as for the canonical stencil (test_gpu_adjoint.py)."""
import ctypes

import numpy as np
import pytest
import torch

import oracle
from hindemith_amd import autograd as AG
from hindemith_amd import synthetic as S
from hindemith_amd._lib import check, lib
from hindemith_amd.kernels import _ptr, stream_ptr

pytestmark = pytest.mark.gpu
TAPS = S.hs_stencil_taps()
_OX, _OY = TAPS["Avg"][1], TAPS["Avg"][2]
_W8 = np.float32([0.11, 0.17, 0.13, 0.19, 0.07, 0.12, 0.05, 0.16])
AVGS = {
    "canonical": TAPS["Avg"],
    "four": (np.full(4, 0.25, np.float32), np.int32([-1, 1, 0, 0]), np.int32([0, 0, -1, 1])),
    "five": (np.float32([0.3, 0.2, 0.25, 0.15, 0.1]), np.int32([0, -1, 1, 0, 0]),
             np.int32([0, 0, 0, -1, 1])),
    "seven": (np.float32([0.1, 0.2, 0.15, 0.15, 0.1, 0.2, 0.1]),
              np.int32([-1, 1, 0, 0, -1, 1, 0]), np.int32([0, 0, -1, 1, -1, 1, 0])),
    "eight": (_W8, np.ascontiguousarray(_OX[::-1]), np.ascontiguousarray(_OY[::-1])),
    "nine": (np.float32([.05, .1, .15, .1, .2, .1, .1, .1, .1]), np.int32([-1, 0, 1] * 3),
             np.repeat(np.int32([-1, 0, 1]), 3)),
}


def _inputs(B, H, W, seed):
    rng = np.random.default_rng(seed)
    prs = [S.hs_pair(H, W, seed=seed * 10 + b) for b in range(B)]
    f = lambda: rng.normal(size=(B, H, W)).astype(np.float32)  # noqa: E731
    return (np.stack([p[0] for p in prs]), np.stack([p[1] for p in prs]),
            rng.uniform(0.5, 2.0, B).astype(np.float32), f(), f())


def _dev(*arrays):
    return [torch.from_numpy(np.ascontiguousarray(a)).cuda() for a in arrays]


@pytest.mark.parametrize("name", [n for n in AVGS if n != "canonical"])
@pytest.mark.parametrize("shape,iters,every", [((2, 40, 52), 30, 7), ((1, 1, 9), 12, 5),
                                               ((1, 9, 1), 12, 5), ((1, 33, 65), 17, 17),
                                               ((2, 100, 130), 10, 3)])
def test_gradient_against_fp64_oracle(name, shape, iters, every):
    taps = dict(TAPS, Avg=AVGS[name])
    I1, I2, al, gu, gv = _inputs(*shape, seed=11)
    t1, t2, ta = (t.requires_grad_(True) for t in _dev(I1, I2, al))
    u, v = AG.horn_schunck(t1, t2, ta, iters=iters, ckpt_every=every, taps=taps)
    got = [t.cpu().numpy() for t in torch.autograd.grad((u, v), (t1, t2, ta), _dev(gu, gv))]
    for b in range(shape[0]):
        ru, rv = oracle.hs_solve(I1[b], I2[b], np.float32(al[b] * al[b]), taps, iters)
        assert np.array_equal(u[b].detach().cpu().numpy(), ru)
        assert np.array_equal(v[b].detach().cpu().numpy(), rv)
        r1, r2, ra, _, _ = oracle.hs_grad(I1[b], I2[b], float(al[b]), taps, iters, gu[b], gv[b])
        for g, r in ((got[0][b], r1), (got[1][b], r2)):
            assert np.linalg.norm(g - r) < 1e-3 * np.linalg.norm(r)
        # (the sum of the terms of both signs that make dL/dalpha is taken against
        # their sizes: their float32 errors do not cancel as they do)
        assert abs(got[2][b] - ra) <= 1e-3 * max(abs(ra), np.linalg.norm(r1))


def _abi(I1, I2, al, gu, gv, taps, iters, every, keep_lin, keep_planes):
    """(u, v, gI1, gI2, galpha) through the C ABI."""
    B, H, W = I1.shape
    L, null = lib(), ctypes.c_void_p(0)
    keep, targs = AG._tap_args(taps)
    u, v = torch.zeros_like(I1), torch.zeros_like(I1)
    nck = L.hmx_hs_ckpt_count(iters, every)
    ck = torch.empty((nck, 2, B, H, W), device="cuda")
    fws = torch.empty(L.hmx_hs_forward_workspace(B, H, W) // 4 + 1, device="cuda")
    last = iters - (nck - 1) * every
    lin = torch.empty((2 * last, B, H, W), device="cuda") if keep_lin else None
    pl = _ptr(lin) if keep_lin else null
    check(L.hmx_hs_forward_ckpt(_ptr(I1), _ptr(I2), B, H, W, _ptr(al), *targs, iters, every,
                                _ptr(u), _ptr(v), _ptr(ck), pl, _ptr(fws), stream_ptr()), "forward")
    g1, g2, ga = torch.empty_like(I1), torch.empty_like(I1), torch.empty_like(al)
    ws = torch.empty(L.hmx_hs_adjoint_workspace_taps(B, H, W, every, *targs[-4:]) // 4 + 1,
                     device="cuda")
    check(L.hmx_hs_adjoint(_ptr(I1), _ptr(I2), B, H, W, _ptr(al), *targs, iters, every, _ptr(ck), pl,
                           _ptr(fws) if keep_planes else null, _ptr(gu), _ptr(gv), _ptr(g1),
                           _ptr(g2), _ptr(ga), null, null, _ptr(ws), stream_ptr()), "adjoint")
    torch.cuda.synchronize()
    return u, v, g1, g2, ga


@pytest.mark.parametrize("name", list(AVGS))
@pytest.mark.parametrize("shape,iters,every", [((2, 100, 200), 37, 10), ((2, 37, 66), 21, 7),
                                               ((1, 40, 52), 8, 8)])
def test_kept_linearisation_matches_recompute_bitwise(name, shape, iters, every):
    """Last segments of 7, 7 and 8 steps.  (The canonical stencil's blocks do not read the
    kept linearisation; its forward writes it all the same.)"""
    taps = dict(TAPS, Avg=AVGS[name])
    args = _dev(*_inputs(*shape, seed=12))
    ref = _abi(*args, taps, iters, every, False, False)
    for keep_lin, keep_planes in ((True, False), (False, True), (True, True)):
        for a, b in zip(ref, _abi(*args, taps, iters, every, keep_lin, keep_planes)):
            assert torch.equal(a, b), (keep_lin, keep_planes)


@pytest.mark.parametrize("name", ["canonical", "five", "nine"])
def test_checkpoint_intervals_agree_bitwise(name):
    """Intervals of one step, of several blocks, of the whole solve and beyond it: the same
    states and sums.  (An interval of 17 runs in blocks of 6, 6 and 5 steps; the
    accumulators' terms are added step by step, however the steps are cut.)"""
    taps = dict(TAPS, Avg=AVGS[name])
    args = _dev(*_inputs(2, 33, 47, seed=13))
    ref = _abi(*args, taps, 25, 8, False, True)
    for every in (1, 6, 9, 17, 25, 40):
        for a, b in zip(ref, _abi(*args, taps, 25, every, False, True)):
            assert torch.equal(a, b), every
