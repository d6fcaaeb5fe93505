"""The sliced CSR's row sums, which read several products ahead: rows of every small
length, and long ones over the boundary of the entries that a work-group takes at once."""
import numpy as np
import pytest
import torch

from hindemith_amd import kernels as K

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("first", [0, 1, 5, 2030, 2041, 2048])
def test_sliced_row_lengths_bitexact(first):
    """Products rounded, then added in entry order; all entries in one slice, whose
    partial sum the empty slices' zeros leave as it is."""
    rng = np.random.default_rng(first)
    lens = np.concatenate([[first], np.arange(40), [700, 3, 0, 2500, 8]])
    N = 8000  # slices of 1000 columns
    nnz = int(lens.sum())
    cols = rng.integers(2000, 3000, nnz).astype(np.int32)
    vals, x = rng.normal(size=nnz).astype(np.float32), rng.normal(size=N).astype(np.float32)
    indptr = np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)
    prod, ref = vals * x[cols], np.zeros(len(lens), np.float32)
    for i in range(len(lens)):
        for p in prod[indptr[i]:indptr[i + 1]]:
            ref[i] = np.float32(ref[i] + p)
    sl = K.CSRSlices(indptr, cols, N, "cuda")
    dev = lambda a: torch.from_numpy(a).cuda()  # noqa: E731
    y = K.csr_spmv_sliced(sl, sl.values(dev(vals)), dev(x))
    assert np.array_equal(y.cpu().numpy(), ref)
