"""Row-register Jacobi variants (hs_rows.h) at the sizes where they can go wrong.

Every variant at the edges of its window: images one row or column narrower and
wider than a tile, the image's last row at every place of a wave's strip (the
row below it is itself), windows that hold the whole image, and k from 1 to the
variant's largest.  Eight distinct weights tell every neighbour apart, and the
fp32 oracle's result is matched bit for bit."""
import numpy as np
import pytest
import torch

import oracle
from hindemith_amd import kernels as K
from hindemith_amd import synthetic as S

pytestmark = pytest.mark.gpu
TAPS = S.hs_stencil_taps()
W8 = np.array([0.11, 0.17, 0.13, 0.19, 0.07, 0.12, 0.05, 0.16], np.float32)
AVG = (W8, TAPS["Avg"][1], TAPS["Avg"][2])  # the canonical offsets and order


def _rows_variants():
    return [(i, v["kmax"]) for i, v in enumerate(K.hs_variants()) if v["kmax"] > 8]


def _inputs(shape, seed):
    rng = np.random.default_rng(seed)
    f = lambda s: (s * rng.normal(size=shape)).astype(np.float32)  # noqa: E731
    return f(0.3), f(0.3), f(0.1), f(1.0), f(1.0)


# heights: 16 k=8 tiles' rows and one more or less, and every remainder of a strip
@pytest.mark.parametrize("shape", [(1, 64), (2, 1), (7, 49), (16, 48), (17, 47), (31, 97),
                                   (33, 63), (50, 65), (64, 129), (81, 33), (150, 62)])
def test_rows_variants_bitexact(shape):
    Ix, Iy, It, u0, v0 = _inputs(shape, shape[0] * 1000 + shape[1])
    dev = lambda a: torch.from_numpy(a).cuda()  # noqa: E731
    dIx, dIy, dIt = dev(Ix), dev(Iy), dev(It)
    variants = _rows_variants()
    assert variants
    for iters in (1, 17):
        ref = oracle.hs_jacobi(Ix, Iy, It, 0.7, AVG, iters, u0, v0)
        for vi, kmax in variants:
            for k in (1, 7, 8, kmax):
                u, v = dev(u0), dev(v0)
                K.hs_jacobi(dIx, dIy, dIt, 0.7, AVG, iters, u, v, variant=vi, k=k)
                assert np.array_equal(u.cpu().numpy(), ref[0]), (vi, k, iters)
                assert np.array_equal(v.cpu().numpy(), ref[1]), (vi, k, iters)


@pytest.mark.parametrize("h", range(20, 33))
def test_rows_last_row_in_every_strip_place(h):
    """den read from an array here (not recomputed), the other form of the prologue."""
    shape = (h, 70)
    Ix, Iy, It, u0, v0 = _inputs(shape, h)
    den = (np.float32(0.7) + Ix * Ix) + Iy * Iy
    ref = oracle.hs_jacobi(Ix, Iy, It, 0.7, AVG, 8, u0, v0)
    dev = lambda a: torch.from_numpy(a).cuda()  # noqa: E731
    for vi, _ in _rows_variants():
        u, v = dev(u0), dev(v0)
        K.hs_jacobi(dev(Ix), dev(Iy), dev(It), 0.0, AVG, 8, u, v, den=dev(den), variant=vi, k=8)
        assert np.array_equal(u.cpu().numpy(), ref[0]), vi
        assert np.array_equal(v.cpu().numpy(), ref[1]), vi


@pytest.mark.parametrize("shape,iters", [((64, 64), 33), ((135, 240), 50), ((301, 517), 23),
                                         ((700, 900), 11), ((1030, 1500), 9)])
def test_default_choice_bitexact(shape, iters):
    """The (variant, k) the sizes pick: one of each class, against a plain sweep."""
    Ix, Iy, It, u0, v0 = (torch.from_numpy(a).cuda() for a in _inputs(shape, iters))
    ru, rv = u0.clone(), v0.clone()
    K.hs_jacobi(Ix, Iy, It, 0.7, AVG, iters, ru, rv, variant=0, k=1)
    u, v = u0.clone(), v0.clone()
    K.hs_jacobi(Ix, Iy, It, 0.7, AVG, iters, u, v)
    assert torch.equal(u, ru) and torch.equal(v, rv)


@pytest.mark.parametrize("taps9", [False, True])
def test_batched_rows_variants_match_single_solves(taps9):
    """The batched row-register variants on uneven pairs, and what they stand for
    with another averaging stencil (variant 8), at even and odd phase counts."""
    from hindemith_amd import batched
    taps = dict(TAPS, Avg=AVG)
    if taps9:
        taps["Avg"] = (np.full(9, 1.0 / 9.0, np.float32), np.array([-1, 0, 1] * 3, np.int32),
                       np.repeat(np.array([-1, 0, 1], np.int32), 3))
    rng = np.random.default_rng(2)
    f = lambda s: torch.from_numpy(rng.normal(size=s).astype(np.float32)).cuda()  # noqa: E731
    shapes = [(1, 70), (33, 47), (90, 131), (64, 49), (257, 3)]
    B = batched.BatchedHS([f(s) for s in shapes], [f(s) for s in shapes], [0.5, 1.0, 1.5, 2.0, 0.75],
                          iters=17, taps=taps)
    ref = [(u.clone(), v.clone()) for u, v in B.solve_each(variant=0, k=1)]
    n = len(batched.batched_variants())
    for vi, k in [(-1, 0)] + [(vi, k) for vi in range(8, n) if vi == 8 or vi >= 12
                              for k in (3, 6, 8)]:
        out = B.run(graph=False, variant=vi, k=k)
        for (u, v), (ru, rv) in zip(out, ref):
            assert torch.equal(u, ru) and torch.equal(v, rv), (vi, k, tuple(u.shape))
