"""Walks through a medium at the queue lengths where their hand-out changes:
one path, the lanes of one wave and one more, the slices of all waves and
claims past them (a wave of samples has width x height x samples_per_wave
paths).  Every sample depends on its pixel and index alone, so the samples of
one wave and of several add up to the same image, but for the rounding of the
sums in double (n additions: n 2^-53 of the sum of positive terms)."""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def cloud():
    import torch

    from sprout_amd import bvh, medium, render, scenes

    assert torch.cuda.is_available(), "GPU tests need a GPU"
    bvh.init(0)
    scene = render.Scene(*scenes.cloud_scene())
    d = scenes.fbm_density(48)
    d[:, :, 30:] *= np.float32(0.2)  # leaves of several sizes
    medium.set_medium(scene, d, *scenes.CLOUD_BOX, scenes.CLOUD_CC_A, scenes.CLOUD_CC_S, scenes.CLOUD_G)
    yield scene
    scene.release()


@pytest.mark.parametrize("spectral", [False, True])
@pytest.mark.parametrize("w,h,spp", [(1, 1, 1), (8, 8, 1), (13, 5, 1), (33, 31, 4), (260, 257, 4)])
def test_waves_of_any_length(cloud, w, h, spp, spectral):
    import torch

    from sprout_amd import render, scenes

    cam = render.camera(w, h, **scenes.CLOUD_CAMERA)
    print(f"{w}x{h}, {spp} samples, spectral {spectral}", flush=True)
    whole, _ = render.render(cloud, cam, 2 * spp, 2 * spp, seed=4, spectral=spectral)
    parts, _ = render.render(cloud, cam, 2 * spp, 1, seed=4, spectral=spectral)
    torch.cuda.synchronize()
    a, b = whole.cpu().numpy(), parts.cpu().numpy()
    assert np.isfinite(a).all() and a.min() >= 0
    assert np.allclose(a, b, rtol=4 * spp * 2.0 ** -53, atol=0)
    if w > 1:
        assert a.max() > 0
