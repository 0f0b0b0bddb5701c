"""Frames through the sample volume (LIC value and field channel in one array)
equal frames from the two volumes bit for bit.  A context makes it once the
frames since the last change of either are worth the pass, so a tiny frame
before a large one reads the volumes and the same frame after it the sample
volume."""
import numpy as np
import pytest

import vectorvisualization_amd as vv
from vectorvisualization_amd import fields

pytestmark = pytest.mark.gpu


def _field(dims, seed):
    rng = np.random.default_rng(seed)
    return rng.normal(size=(dims[2], dims[1], dims[0], 3)).astype(np.float32)


def _cams(ctx):
    ext, _, cen = ctx.field_geometry()
    return (fields.orbit_camera(9, 7, cen, 0.7, 0.4), fields.orbit_camera(300, 260, cen, -0.5, 0.3))


def _same(ctx, adjoint=False):
    """The small frame (and its adjoint) before and after the large one."""
    small, large = _cams(ctx)
    out = []
    for _ in range(2):
        got = [ctx.render(small)]
        if adjoint:
            got.append(ctx.render_record(small))
            d = np.random.default_rng(2).normal(size=small.width * small.height * 4).astype(np.float32)
            got += list(ctx.render_adjoint(small, d))
        out.append(got)
        ctx.render(large)
    assert np.max(out[0][0]) > 0
    for a, b in zip(*out):
        assert np.array_equal(a, b)


@pytest.mark.parametrize("storage", [vv.STORE_FP32, vv.STORE_FP16, vv.STORE_UNORM8])
@pytest.mark.parametrize("dims,spacing", [((40, 33, 37), (1.0, 1.0, 1.0)), ((41, 24, 40), (1.0, 1.5, 2.0)),
                                          ((36, 40, 44), (0.5, 1.0, 0.7))])
def test_frames_equal(ctx, storage, dims, spacing):
    ctx.upload_field(_field(dims, 1), dims, spacing=spacing, storage=storage)
    ctx.generate_noise(3, vv.NOISE_UNIFORM, 0.0, dims)
    p = vv.default_lic_params()
    p.steps_forward = p.steps_backward = 4
    p.gradient_scale = 4.0
    ctx.set_lic_params(p)
    ctx.set_tf(*fields.tf_magnitude(0.05, 0.2))
    ctx.compute_lic()
    _same(ctx, adjoint=True)
    # another TF channel, an opacity scale, another field and another LIC
    # volume: each drops the sample volume
    p.tf_index = vv.TF_INDEX_MAG
    ctx.set_lic_params(p)
    _same(ctx)
    ctx.set_opacity_scale(np.random.default_rng(5).uniform(0.5, 1.5, dims[0] * dims[1] * dims[2]).astype(np.float32))
    _same(ctx, adjoint=True)
    ctx.upload_field(_field(dims, 9), dims, spacing=spacing, storage=storage)
    _same(ctx)
    ctx.upload_lic(np.random.default_rng(6).uniform(0.0, 2.0, dims[0] * dims[1] * dims[2]).astype(np.float32), 1, dims)
    _same(ctx)


def test_stale_sample_volume_is_not_read(ctx):
    """A frame after each change equals the frame of a fresh context."""
    dims = (32, 32, 32)

    def load(c, seed, index):
        c.upload_field(_field(dims, seed), dims)
        c.generate_noise(seed, vv.NOISE_UNIFORM, 0.0, dims)
        p = vv.default_lic_params()
        p.steps_forward = p.steps_backward = 3
        p.tf_index = index
        c.set_lic_params(p)
        c.compute_lic()

    for seed, index in ((1, vv.TF_INDEX_B), (2, vv.TF_INDEX_B), (2, vv.TF_INDEX_MAG), (3, vv.TF_INDEX_B)):
        load(ctx, seed, index)
        with vv.Context(0) as fresh:
            load(fresh, seed, index)
            for cam in _cams(ctx)[::-1]:
                assert np.array_equal(ctx.render(cam), fresh.render(cam))


@pytest.mark.parametrize("bad", [np.nan, np.inf, -np.inf, 3e38])
def test_groups_with_values_that_are_not_finite(ctx, bad):
    """Samples that are not finite reach the image as with one lane per pixel
    (the grouped casters clamp finite rounds with the hardware's modifier,
    which would drop a NaN)."""
    dims = (24, 24, 24)
    ctx.upload_field(_field(dims, 4), dims)
    lic = np.random.default_rng(8).uniform(0.0, 1.0, (24, 24, 24)).astype(np.float32)
    lic[12:, 5:9, 7] = bad
    lic[3, 4, 20:] = -bad
    ctx.upload_lic(lic, 1, dims)
    ctx.set_tf(*fields.tf_magnitude(0.05, 0.3))
    cam = _cams(ctx)[1]
    cam.width, cam.height = 61, 47
    img = {}
    for G in (1, 2, 4, 8, 16, 32):
        ctx.set_tuning("render.volume_group", G)
        img[G] = ctx.render(cam, count_samples=True)
    for G, (im, n) in img.items():
        np.testing.assert_array_equal(im, img[1][0], err_msg=str(G))
        assert n == img[1][1]


@pytest.mark.parametrize("storage", [vv.STORE_FP32, vv.STORE_FP16, vv.STORE_UNORM8])
@pytest.mark.parametrize("dims,spacing", [((40, 33, 37), (1.0, 1.5, 2.0)), ((36, 40, 44), (0.5, 1.0, 0.7))])
def test_rgba_frames_equal(ctx, storage, dims, spacing):
    """An RGBA LIC volume with the field's channel from its plane."""
    ctx.upload_field(_field(dims, 1), dims, spacing=spacing, storage=storage)
    ctx.generate_noise(3, vv.NOISE_UNIFORM, 0.0, dims, with_gradients=True)
    p = vv.default_lic_params()
    p.steps_forward = p.steps_backward = 4
    p.gradient_scale = 4.0
    p.illum_mode = vv.ILLUM_GRADIENT
    ctx.set_lic_params(p)
    ctx.set_tf(*fields.tf_magnitude(0.05, 0.2))
    ctx.compute_lic()
    _same(ctx, adjoint=True)
    p.tf_index = vv.TF_INDEX_MAG
    ctx.set_lic_params(p)
    _same(ctx)
    ctx.set_opacity_scale(np.random.default_rng(5).uniform(0.5, 1.5, dims[0] * dims[1] * dims[2]).astype(np.float32))
    _same(ctx, adjoint=True)
    ctx.upload_field(_field(dims, 2), dims, spacing=spacing, storage=storage)
    _same(ctx)
