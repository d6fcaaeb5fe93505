"""The one-lane CSR's passes over a wave's entries: one build per number of 64-entry chunks."""
import numpy as np
import pytest
import torch

import oracle
from hindemith_amd import kernels as K

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("span", [n for c in range(1, 11) for n in (64 * c - 1, 64 * c, 64 * c + 1)])
def test_csr_one_lane_every_chunk_count_bitexact(span):
    """The entries of a wave lie in few of its rows, or one; the last wave is short."""
    rng = np.random.default_rng(span)
    rows, N = 150, 901
    per = np.zeros(rows, np.int64)
    for w in range(0, rows, 64):
        own = rng.integers(w, min(w + 64, rows), 5)
        np.add.at(per, own[rng.integers(0, 5, span)], 1)
    indptr = np.concatenate([[0], np.cumsum(per)]).astype(np.int32)
    indices = rng.integers(0, N, int(indptr[-1])).astype(np.int32)
    data = rng.normal(size=len(indices)).astype(np.float32)
    x = rng.normal(size=N).astype(np.float32)
    dev = lambda a: torch.from_numpy(a).cuda()  # noqa: E731
    y = K.csr_spmv(dev(indptr), dev(indices), dev(data), dev(x), lanes_per_row=1)
    assert np.array_equal(y.cpu().numpy(), oracle.csr_spmv(indptr, indices, data, x))
