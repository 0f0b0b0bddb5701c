"""The one-pass gradient noise texture has the oracle's bytes at the edges of
its tiles (32 x 8 voxels, columns of 4 or 16 slices) and windows: volumes of
two and three texels, one short of, at and past a tile, and one large enough
for the long columns."""
import numpy as np
import pytest

import vectorvisualization_amd as vv
from oracle import oracle as orc

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dims", [(2, 2, 2), (3, 4, 5), (5, 3, 2), (31, 7, 3), (32, 8, 4), (33, 9, 5), (66, 17, 13),
                                  (200, 200, 131)])
@pytest.mark.parametrize("kind,density", [(vv.NOISE_BINARY, 0.2), (vv.NOISE_UNIFORM, 0.0)])
def test_texture_bytes(ctx, dims, kind, density):
    ctx.generate_noise(11, kind, density, dims, with_gradients=True)
    got = ctx.download_noise().reshape(-1, 4)
    n = orc.gen_noise(11, kind, density, dims)
    np.testing.assert_array_equal(got[:, 3], n)
    np.testing.assert_array_equal(got[:, :3], orc.noise_gradients(n, dims).reshape(-1, 3))
