"""WarpImg2D from a megapixel on, four rows per thread: heights that leave 1 to 3 rows
over, a single column block, and more row groups than the grid has."""
import numpy as np
import pytest
import torch

import oracle
from hindemith_amd import kernels as K

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape", [(1021, 1027), (1026, 1025), (1, 1 << 20), (2, 600001),
                                   (349527, 3), (262149, 4), (1023, 1025)])
def test_warp_rows_bitexact(shape):
    rng = np.random.default_rng(shape[0])
    src, ox, oy = (rng.normal(size=shape).astype(np.float32) for _ in range(3))
    ox, oy = 4 * ox, 4 * oy
    ox.flat[::17] = np.round(ox.flat[::17])
    oy.flat[::29] = 1e6
    got = K.warp_img2d(*(torch.from_numpy(a).cuda() for a in (src, ox, oy))).cpu().numpy()
    assert np.array_equal(got, oracle.warp_img2d(src, ox, oy))
