"""LIC with RGBA noise, the scalar gate and SPEED_OF_FLOW through the per-lane
cell caches gives the bits of the kernels without them ("lic.cache" 0), for
the LIC volume and the on-the-fly casters: two texels on an axis, noise on and
off the field's grid, a gate volume of other dims, steps that jump several
cells, leave the volume or end a hundred million volumes away."""
import numpy as np
import pytest
import torch

import vectorvisualization_amd as vv
from vectorvisualization_amd import fields

pytestmark = pytest.mark.gpu


def _scene(ctx, dims, storage, kind, h, speed):
    v = np.zeros((dims[2], dims[1], dims[0], 3), np.float32)
    z, y, x = np.meshgrid(*(np.linspace(0.0, 1.0, n) for n in dims[::-1]), indexing="ij")
    v[..., 0], v[..., 1], v[..., 2] = 1.0 + 0.3 * y, 0.5 * np.cos(2.0 * x), 0.7 - z
    ctx.upload_field(v, dims, storage=storage)
    ndims = (7, 4, 5) if kind == "rgba_off" else dims
    ctx.generate_noise(5, vv.NOISE_UNIFORM, 0.0, ndims, with_gradients=kind.startswith("rgba"))
    p = vv.default_lic_params()
    p.steps_forward, p.steps_backward, p.step_size_lic, p.freq_scale = 9, 6, h, 1.5
    p.speed_of_flow = speed
    if kind == "gate":
        sdims = (5, 3, 6)
        rng = np.random.default_rng(3)
        ctx.upload_scalar(rng.integers(0, 256, sdims[::-1], dtype=np.uint8), sdims)
        p.gate_enable, p.gate_lo, p.gate_hi = 1, 0.3, 0.8
    ctx.set_lic_params(p)
    ctx.set_tf(*fields.tf_magnitude())
    return p


def _both(ctx, fn):
    out = []
    for cache in (0, 1):
        ctx.set_tuning("lic.cache", cache)
        out.append(fn())
    return out


@pytest.mark.parametrize("dims", [(2, 2, 2), (9, 2, 33), (13, 11, 7)])
@pytest.mark.parametrize("storage", [vv.STORE_FP32, vv.STORE_FP16, vv.STORE_UNORM8])
@pytest.mark.parametrize("kind,speed", [("rgba", 0), ("rgba_off", 0), ("gate", 0), ("rgba", 1), ("rgba_off", 1),
                                        ("gate", 1), ("plain", 1)])
@pytest.mark.parametrize("h", [0.01, 0.5, 1e8])
def test_volume_bits(ctx, dims, storage, kind, speed, h):
    _scene(ctx, dims, storage, kind, h, speed)

    def lic():
        ctx.compute_lic()
        return ctx.download_lic()

    a, b = _both(ctx, lic)
    assert np.abs(a).max() > 0
    np.testing.assert_array_equal(a, b)


@pytest.mark.parametrize("storage", [vv.STORE_FP32, vv.STORE_FP16, vv.STORE_UNORM8])
@pytest.mark.parametrize("kind", ["rgba", "rgba_off", "gate"])
@pytest.mark.parametrize("group", [0, 1, 4])
def test_on_the_fly_bits(ctx, storage, kind, group):
    p = _scene(ctx, (13, 11, 7), storage, kind, 0.03, 0)
    p.step_size_vol = 1 / 32
    ctx.set_lic_params(p)
    ctx.set_tuning("render.ray_group", group)
    cam = fields.orbit_camera(37, 21, (0.5, 0.5, 0.5), 0.4, 0.3)
    for render in (ctx.render_fused, ctx.render_slices):
        a, b = _both(ctx, lambda: render(cam))
        assert np.abs(np.asarray(a)).max() > 0
        np.testing.assert_array_equal(np.asarray(a), np.asarray(b))


def test_captured_lic_reads_later_fields(ctx):
    """A captured LIC with RGBA noise is the LIC of the field at each replay."""
    dims = (13, 11, 7)
    _scene(ctx, dims, vv.STORE_FP32, "rgba", 0.03, 0)
    ctx.compute_lic()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=ctx._torch_stream()):
        ctx.compute_lic()
    for seed in (1, 2):
        v = np.random.default_rng(seed).normal(size=dims[::-1] + (3,)).astype(np.float32)
        ctx.upload_field(v, dims)
        g.replay()
        torch.cuda.synchronize()
        got = ctx.download_lic()
        ctx.compute_lic()
        np.testing.assert_array_equal(got, ctx.download_lic())


@pytest.mark.parametrize("storage,kind,steps,size", [
    (st, kind, steps, size)
    for st, kind, edges in ((vv.STORE_FP32, "gate", ((4, 3), (4, 4), (12, 12), (13, 12))),
                            (vv.STORE_UNORM8, "gate", ((4, 3), (4, 4), (12, 12), (13, 12))),
                            (vv.STORE_FP16, "rgba", ((6, 5), (6, 6), (22, 22), (23, 22))))
    for steps, size in zip(edges, ((149, 111), (149, 111), (300, 261), (300, 261)))])
@pytest.mark.parametrize("group", [1, 4])
def test_slices_of_short_and_longer_streamlines(ctx, storage, kind, steps, size, group):
    """Slices on both sides of the lengths from which they take the caches."""
    p = _scene(ctx, (13, 11, 7), storage, kind, 0.03, 0)
    p.step_size_vol = 1 / 32
    p.steps_forward, p.steps_backward = steps
    ctx.set_lic_params(p)
    ctx.set_tuning("render.ray_group", group)
    cam = fields.orbit_camera(*size, (0.5, 0.5, 0.5), 0.4, 0.3)
    a, b = _both(ctx, lambda: ctx.render_slices(cam))
    assert np.abs(a).max() > 0
    np.testing.assert_array_equal(a, b)
