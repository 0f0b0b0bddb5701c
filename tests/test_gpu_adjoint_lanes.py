"""The recorded frame of a large view takes fewer lanes per ray than the
backward walk: image and gradients keep the bits of four lanes for both."""
import numpy as np
import pytest

import vectorvisualization_amd as vv
from vectorvisualization_amd import fields

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("w,h", [(723, 725), (724, 725), (800, 701), (1254, 1254), (1256, 1253), (1301, 1250)])
def test_gradients_equal(ctx, w, h):
    dims = (24, 20, 28)
    rng = np.random.default_rng(4)
    ctx.upload_field(rng.normal(size=dims[::-1] + (3,)).astype(np.float32), dims)
    ctx.generate_noise(3, vv.NOISE_UNIFORM, 0.0, dims)
    p = vv.default_lic_params()
    p.steps_forward = p.steps_backward = 4
    p.gradient_scale, p.step_size_vol = 4.0, 1 / 48
    ctx.set_lic_params(p)
    ctx.set_tf(*fields.tf_magnitude(0.05, 0.2))
    ctx.compute_lic()
    ctx.set_opacity_scale(rng.uniform(0.5, 1.5, dims[0] * dims[1] * dims[2]).astype(np.float32))
    cam = fields.orbit_camera(w, h, ctx.field_geometry()[2], 0.7, 0.4)
    d = rng.normal(size=w * h * 4).astype(np.float32)
    out = []
    for group in (4, 0):
        ctx.set_tuning("render.volume_group", group)
        out.append([ctx.render_record(cam), *ctx.render_adjoint(cam, d), *ctx.render_adjoint(cam, d)])
    assert np.abs(out[0][1]).max() > 0 and np.abs(out[0][2]).max() > 0
    for a, b in zip(*out):
        np.testing.assert_array_equal(a, b)
