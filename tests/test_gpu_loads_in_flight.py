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


@pytest.mark.parametrize("n", [0, 1, 511, 512, 513, 1535, 2047, 2048, 2049, 4097])
@pytest.mark.parametrize("rows", [1, 512, 515])
def test_csr_sliced_chunk_edges_bitexact(n, rows):
    """n entries of one column slice in the first 512 rows, around the entries a
    work-group takes at once (one row holds a third of them), one entry per row in
    another slice: products rounded, then added in entry order, slices in order."""
    rng = np.random.default_rng(n * 7 + rows)
    N = 8000  # slices of 1000 columns
    near = min(rows, 512)
    lens = np.bincount(rng.integers(0, near, n - n // 3), minlength=rows)
    lens[near // 2] += n // 3
    cols, vals, ref = [], [], np.zeros(rows, np.float32)
    x = rng.normal(size=N).astype(np.float32)
    for i in range(rows):
        c = np.concatenate([rng.integers(3000, 4000, lens[i]), rng.integers(7000, N, 1)])
        v = rng.normal(size=len(c)).astype(np.float32)
        part = np.float32(0)
        for p in v[:-1] * x[c[:-1]]:
            part = np.float32(part + p)
        ref[i] = np.float32(part + np.float32(v[-1] * x[c[-1]]))
        cols.append(c)
        vals.append(v)
    indptr = np.concatenate([[0], np.cumsum(lens + 1)]).astype(np.int32)
    sl = K.CSRSlices(indptr, np.concatenate(cols).astype(np.int32), N, "cuda")
    y = K.csr_spmv_sliced(sl, sl.values(dev(np.concatenate(vals))), dev(x))
    assert np.array_equal(y.cpu().numpy(), ref)
