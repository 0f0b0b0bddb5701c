"""The ray casters' sample volume against the two volumes it is made of, switched
by "render.sample_volume": with an opacity scale, on stretched boxes, past
2 GiB, and where a captured graph rewrites what it was made of."""
import numpy as np
import pytest
import torch

import vectorvisualization_amd as vv
from vectorvisualization_amd import fields

pytestmark = pytest.mark.gpu


def _field(dims, seed):
    return np.random.default_rng(seed).normal(size=dims[::-1] + (3,)).astype(np.float32)


def _scene(ctx, dims, seed, grad=False, storage=vv.STORE_FP32, spacing=(1.0, 1.0, 1.0), ndims=None):
    ctx.upload_field(_field(dims, seed), dims, spacing=spacing, storage=storage)
    ctx.generate_noise(seed, vv.NOISE_UNIFORM, 0.0, ndims or dims, with_gradients=grad)
    p = vv.default_lic_params()
    p.steps_forward = p.steps_backward = 4
    p.gradient_scale = 4.0
    p.illum_mode = vv.ILLUM_GRADIENT if grad else vv.ILLUM_LIC
    ctx.set_lic_params(p)
    ctx.set_tf(*fields.tf_magnitude(0.05, 0.2))
    return p


def _cams(ctx):
    cen = ctx.field_geometry()[2]
    return fields.orbit_camera(300, 260, cen, -0.5, 0.3), fields.orbit_camera(29, 31, cen, 0.7, 0.4)


@pytest.mark.parametrize("grad", [False, True])
def test_captured_lic_and_frame(ctx, grad):
    """A graph of vv_compute_lic and of a frame, recorded after the sample volume
    was made, and plain frames between its replays: those of a new context."""
    dims, ndims = (33, 28, 31), (16, 16, 16)
    p = _scene(ctx, dims, 1, grad, ndims=ndims)
    ctx.compute_lic()
    cam = _cams(ctx)[0]
    image = torch.empty((cam.height, cam.width, 4), device="cuda")
    for _ in range(2):
        ctx.render(cam, out=image)
    ctx.synchronize()
    assert ctx.get_tuning("render.sample_volume") == 1
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=ctx._torch_stream()):
        assert vv.LIB.vv_render(ctx.handle, vv._lib.C.byref(cam), image.data_ptr(), 1, None) == 0
        assert ctx.get_tuning("render.sample_volume") == 1
        ctx.compute_lic()
        assert vv.LIB.vv_render(ctx.handle, vv._lib.C.byref(cam), image.data_ptr(), 1, None) == 0
    assert ctx.get_tuning("render.sample_volume") == 0
    for seed in (2, 3):
        ctx.upload_field(_field(dims, seed), dims)
        ctx.render(cam)  # the new field with the old LIC volume
        g.replay()
        torch.cuda.synchronize()
        got, plain = image.cpu().numpy().ravel(), ctx.render(cam)
        with vv.Context(0) as fresh:
            _scene(fresh, dims, 1, grad, ndims=ndims)
            fresh.upload_field(_field(dims, seed), dims)
            fresh.set_lic_params(p)
            fresh.compute_lic()
            want = fresh.render(cam)
        assert np.max(want) > 0
        np.testing.assert_array_equal(got, want)
        np.testing.assert_array_equal(plain, want)


def _off_and_on(ctx, load, draw):
    """draw() from the two volumes and through the sample volume, which frames of
    this size have made by then."""
    large = _cams(ctx)[0]
    out = []
    for on in (0, 1):
        ctx.set_tuning("render.sample_volume", on)
        load()
        for _ in range(2):
            ctx.render(large)
        out.append(draw())
    for a, b in zip(*out):
        assert np.any(a != 0)
        np.testing.assert_array_equal(a, b)


@pytest.mark.parametrize("storage", [vv.STORE_FP32, vv.STORE_FP16, vv.STORE_UNORM8])
@pytest.mark.parametrize("dims,spacing", [((40, 33, 37), (1.0, 1.0, 1.0)), ((36, 40, 44), (1.3, 1.0, 1.1))])
@pytest.mark.parametrize("grad", [False, True])
@pytest.mark.parametrize("index", [vv.TF_INDEX_B, vv.TF_INDEX_MAG])
def test_opacity_scale(ctx, storage, dims, spacing, grad, index):
    """Frame, recorded frame and both gradients with an opacity scale."""
    p = _scene(ctx, dims, 4, grad, storage, spacing)
    p.tf_index = index
    ctx.set_lic_params(p)
    cam = _cams(ctx)[1]
    sigma = np.random.default_rng(5).uniform(0.5, 1.5, dims[0] * dims[1] * dims[2]).astype(np.float32)
    dimg = np.random.default_rng(6).normal(size=cam.width * cam.height * 4).astype(np.float32)

    def load():
        ctx.compute_lic()
        ctx.set_opacity_scale(sigma)

    def draw():
        return [ctx.render(cam), ctx.render_record(cam), *ctx.render_adjoint(cam, dimg)]

    _off_and_on(ctx, load, draw)


def test_past_2gib(ctx):
    """A sample volume of 3.4 GB, read with 32-bit byte offsets."""
    dims = (1024, 1024, 400)
    assert 2 ** 31 < 8 * (dims[0] + 2) * (dims[1] + 2) * (dims[2] + 2) < 2 ** 32
    z = torch.linspace(0.0, 9.0, dims[2], device="cuda").view(-1, 1, 1)
    y = torch.linspace(0.0, 7.0, dims[1], device="cuda").view(1, -1, 1)
    x = torch.linspace(0.0, 5.0, dims[0], device="cuda").view(1, 1, -1)
    v = torch.empty(dims[::-1] + (3,), device="cuda")
    v[..., 0], v[..., 1], v[..., 2] = torch.sin(z) + 0 * y + 0 * x, torch.cos(x) + 0 * y + 0 * z, torch.sin(y) * z + 0 * x
    ctx.upload_field(v, dims, storage=vv.STORE_UNORM8)
    del v
    lic = torch.rand(dims[::-1], device="cuda", generator=torch.Generator(device="cuda").manual_seed(3))
    p = vv.default_lic_params()
    p.step_size_vol, p.num_iterations = 1.0 / 1024.0, 64
    ctx.set_lic_params(p)
    ctx.set_tf(*fields.tf_magnitude(0.02, 0.01))
    cen = ctx.field_geometry()[2]
    frames = []
    for on in (0, 1):
        ctx.set_tuning("render.sample_volume", on)
        ctx.upload_lic(lic, 1, dims)
        cams = [fields.orbit_camera(1024, 1024, cen, yaw, pitch) for yaw, pitch in ((0.4, 0.3), (2.8, -0.3))]
        frames.append([ctx.render(c).copy() for c in cams])
    for a, b in zip(*frames):
        assert np.max(a) > 0.01
        np.testing.assert_array_equal(a, b)
