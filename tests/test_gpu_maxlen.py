"""The largest vector length of an upload, read four vectors at a time from
aligned arrays and one at a time from others, scales the magnitude channel as
in float64: voxel counts with every remainder, the largest vector first and
last, and a field interpolated between two."""
import numpy as np
import pytest
import torch

import vectorvisualization_amd as vv

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dims", [(2, 2, 2), (3, 3, 3), (5, 5, 2), (7, 5, 3), (111, 70, 150)])
@pytest.mark.parametrize("offset", [0, 1])
@pytest.mark.parametrize("last", [False, True])
@pytest.mark.parametrize("lerp", [False, True])
def test_magnitudes(ctx, dims, offset, last, lerp):
    n = dims[0] * dims[1] * dims[2]
    rng = np.random.default_rng(n)
    v = [rng.normal(size=(n, 3)).astype(np.float32) for _ in range(2)]
    for a in v:
        a[-1 if last else 0] = (30.0, 40.0, 5.0)
    buf = [torch.zeros(3 * n + offset, device="cuda:0") for _ in v]
    dev = [b[offset:] for b in buf]
    for d, a in zip(dev, v):
        d.copy_(torch.from_numpy(a.ravel()))
    if lerp:
        ctx.upload_field(dev[0], dims, v1=dev[1], lerp_t=0.25)
        t = v[0] + np.float32(0.25) * (v[1] - v[0])
    else:
        ctx.upload_field(dev[0], dims)
        t = v[0]
    got = ctx.download_field(dims).reshape(-1, 4)[:, 3]
    length = np.sqrt(np.sum(t.astype(np.float64) ** 2, axis=1))
    np.testing.assert_allclose(got, length / length.max(), rtol=0, atol=1e-6)
