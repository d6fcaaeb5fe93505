"""HSMatrixPowers where its outputs leave the chip by non-temporal stores (rows on
64-byte sectors, powers beyond 128 MB), several launches of powers included, and
the tile and strip edges of its window; bit for bit against the fp32 oracle."""
import numpy as np
import pytest
import torch

import oracle
from hindemith_amd import kernels as K

pytestmark = pytest.mark.gpu


def _check(H, W, steps, scale=0.3):
    rng = np.random.default_rng(H * 31 + W + steps)
    g = [(scale * rng.normal(size=(H, W))).astype(np.float32) for _ in range(4)]
    V0, V1 = K.hs_matrix_powers(0.15, *(torch.from_numpy(a).cuda() for a in g), steps)
    R0, R1 = oracle.hs_matrix_powers(0.15, *g, steps)
    for s in range(steps):
        assert np.array_equal(V0[s].cpu().numpy(), R0[s]), s
        assert np.array_equal(V1[s].cpu().numpy(), R1[s]), s


@pytest.mark.parametrize("shape,steps", [((1000, 1936), 9), ((32767, 16), 33), ((333, 3200), 17)])
def test_powers_large_outputs_bitexact(shape, steps):
    assert 2 * steps * shape[0] * shape[1] * 4 >= 1 << 27
    _check(*shape, steps)


@pytest.mark.parametrize("H", [1, 3, 4, 5, 47, 48, 49, 56, 57, 97])
@pytest.mark.parametrize("W", [1, 47, 48, 49, 56, 57, 97])
def test_powers_tile_edges_bitexact(H, W):
    _check(H, W, 9)


@pytest.mark.parametrize("steps", [2, 3, 8, 9, 10])
def test_powers_counts_at_tile_edges_bitexact(steps):
    """Fewer powers per launch leave more rows of a window to its tile."""
    _check(64 - 2 * (steps - 1) % 16 + 50, 99, steps)
