"""The tile order of the LIC kernels: on grids that no tile or super-tile
divides, every voxel is computed once, whatever the super-tile's shape."""
import numpy as np
import pytest

import vectorvisualization_amd as vv
from oracle import oracle as orc

from conftest import rel_err

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("tile", [(16, 4, 4), (4, 4, 16), (1, 1, 256), (256, 1, 1)])
@pytest.mark.parametrize("sup", [(2, 16, 16), (1, 2, 8), (4, 1, 2), (256, 256, 256)])
def test_tile_order_covers_odd_grids(ctx, tile, sup):
    dims = (37, 21, 18)
    rng = np.random.default_rng(7)
    v = rng.normal(size=(dims[2], dims[1], dims[0], 3)).astype(np.float32)
    ctx.upload_field(v, dims)
    ctx.generate_noise(3, vv.NOISE_UNIFORM, 0.0, dims)
    p = vv.default_lic_params()
    p.steps_forward = p.steps_backward = 5
    ctx.set_lic_params(p)
    for k, t, s in zip("xyz", tile, sup):
        ctx.set_tuning("lic.tile_" + k, t)
        ctx.set_tuning("lic.super_" + k, s)
    # stale values would show where a voxel is missed
    ctx.upload_lic(np.full(dims[0] * dims[1] * dims[2], 7.0, np.float32), 1, dims)
    ctx.compute_lic()
    lic = ctx.download_lic()
    op = orc.params(steps_forward=5, steps_backward=5)
    ref = orc.lic(orc.encode_field(v, dims), dims, orc.gen_noise(3, vv.NOISE_UNIFORM, 0.0, dims), 1, dims,
                  np.full(256, 255, np.uint8), op, scale=ctx.field_geometry()[1])
    assert rel_err(lic, ref) <= 1e-5
