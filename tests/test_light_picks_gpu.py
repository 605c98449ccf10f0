"""Light picks made apart from their splitting descent, against the oracle's
one descent, at the tree sizes where it changes: one light, one leaf (2 and 4
lights), the first inner node, and enough bright lights that the descent ends
at the 64 picks a vertex may have; and the renderer's vertices on the same
scenes, same random numbers."""

import numpy as np
import pytest

from oracle import oracle as O
from scene_util import light_tree

pytestmark = pytest.mark.gpu

F = np.float32


def scene_of(n, radiance):
    from sprout_amd import scenes

    rng = np.random.default_rng(n)
    mats = np.zeros(1 + n, scenes.MATERIAL_DTYPE)
    mats["color"][0] = 0.7
    mats["kind"][1:] = scenes.LIGHT
    mats["emission"][1:] = rng.uniform(0.5, 1.0, (n, 3)) * radiance * np.exp(2 * rng.normal(size=(n, 1)))
    c = rng.uniform((-1, 1.2, -1), (1, 2, 1), (n, 3))
    e = rng.uniform(0.02, 0.1, (n, 1, 1)) * np.array([[0, 0, 0], [1, 0, 0], [0, 0, 1]])
    tris = c[:, None] + e
    pos = np.concatenate([np.array([[-3, 0, -3], [-3, 0, 3], [3, 0, 3], [3, 0, -3]]),
                          tris.reshape(-1, 3)]).astype(F)
    idx = np.concatenate([[[0, 1, 2], [0, 2, 3]], 4 + np.arange(3 * n).reshape(-1, 3)]).astype(np.uint32)
    tmat = np.concatenate([[0, 0], 1 + np.arange(n)]).astype(np.uint32)
    return pos, idx, tmat, mats


@pytest.mark.parametrize("n,radiance", [(1, 5), (2, 5), (4, 5000), (5, 5000), (40, 5), (300, 1e6)])
@pytest.mark.parametrize("split", [False, True])
def test_picks_of_trees_of_any_size(n, radiance, split):
    import torch

    from sprout_amd import bvh, lights, render

    assert torch.cuda.is_available(), "GPU tests need a GPU"
    bvh.init(0)
    scene = scene_of(n, radiance)
    sc = render.Scene(*scene)
    tree = light_tree(*scene)
    rng = np.random.default_rng(5)
    m = 150
    p = rng.uniform((-1, 0, -1), (1, 2, 1), (m, 3)).astype(F)
    nrm = rng.normal(size=(m, 3))
    nrm = (nrm / np.linalg.norm(nrm, axis=1, keepdims=True)).astype(F)
    u = rng.random(m).astype(F)
    print(f"{n} lights, split {split}", flush=True)
    picks, pdfs, counts = lights.sample(sc, p, nrm, u, split)
    for k in range(m):
        ls, ps = tree.random_light(p[k], nrm[k], float(u[k]), split)
        assert counts[k] == len(ls)
        assert np.array_equal(picks[k, :len(ls)], ls)
        assert np.allclose(pdfs[k, :len(ls)], ps, rtol=1e-5, atol=0)
    if split and n == 300:
        assert counts.max() > 16
    w, h, spp = 24, 16, 2
    view = dict(eye=(0.0, 1.5, 4.0), target=(0.0, 0.5, 0.0), up=(0.0, 1.0, 0.0), fov_deg=45.0)
    img, _ = render.render(sc, render.camera(w, h, **view), spp, 2, seed=6)
    torch.cuda.synchronize()
    img = img.cpu().numpy() / spp
    ref = O.render(*scene, w, h, spp, view, tree, seed=6) / spp
    sc.release()
    # the device's and the host's trigonometry differ in the last bit, which
    # turns single decisions of few paths: nearly every pixel is the same
    diff = np.abs(img - ref) / np.maximum(ref, 1e-3 * ref.max())
    assert ref.max() > 0 and np.mean(diff < 1e-3) > 0.97
