"""The sizes at which loops with several reads in flight per thread change branch:
the one-lane CSR's spans around its unrolled read and its LDS share, and the
sum's element counts around one unrolled step of its grid."""
import numpy as np
import pytest
import torch

import oracle
from hindemith_amd import kernels as K

pytestmark = pytest.mark.gpu


def dev(a):
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


@pytest.mark.parametrize("span", [0, 1, 63, 64, 65, 319, 320, 321, 639, 640, 641, 1000])
@pytest.mark.parametrize("rows", [64, 65, 200])
def test_csr_one_lane_spans_bitexact(span, rows):
    """64 consecutive rows hold `span` entries (a row's share differs by at most
    one); the last row of all ends the arrays, so a read past a span shows as a
    wrong value or an index of another row."""
    rng = np.random.default_rng(span * 1000 + rows)
    per = np.array([span // 64 + (i % 64 < span % 64) for i in range(rows)])
    indptr = np.concatenate([[0], np.cumsum(per)]).astype(np.int32)
    nnz, N = int(indptr[-1]), 777
    indices = rng.integers(0, N, nnz).astype(np.int32)
    data = rng.normal(size=nnz).astype(np.float32)
    x = rng.normal(size=N).astype(np.float32)
    y = K.csr_spmv(dev(indptr), dev(indices), dev(data), dev(x), lanes_per_row=1)
    assert np.array_equal(y.cpu().numpy(), oracle.csr_spmv(indptr, indices, data, x))


@pytest.mark.parametrize("n", [1, 255, 257, 7 * 262144 + 1, 8 * 262144 - 1, 8 * 262144,
                               8 * 262144 + 1, 15 * 262144 + 300, 16 * 262144 + 5])
def test_sum_unroll_edges(n):
    """Every element counts once: integers, whose sum float64 holds exactly, then
    one rounding to float32."""
    x = np.random.default_rng(n).integers(-8, 9, n).astype(np.float32)
    x[-1] = 5.0
    got = K.sum2d(dev(x)).cpu().numpy()
    assert got[0] == np.float32(x.sum(dtype=np.float64))
