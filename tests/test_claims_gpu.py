"""Counters that no kernel of their own clears: ray claims across launches
that use them and launches whose waves' slices hold all rays, in every order,
and the queues, totals and claims of a frame's bounces, launched kernel by
kernel, captured, replayed and regenerating, after one another."""

import numpy as np
import pytest

from oracle import oracle as O

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def gpu():
    import torch

    from sprout_amd import bvh

    assert torch.cuda.is_available(), "GPU tests need a GPU"
    bvh.init(0)
    yield bvh
    torch.cuda.synchronize()


def test_launches_after_one_another(gpu):
    """2^19 rays fill the slices of the resident grid of 256 CUs: launches on
    either side of it, and small ones between, against the same rays traced
    in small launches"""
    import torch

    from sprout_amd import scenes

    pos, idx = scenes.displaced_icosphere(subdivisions=2, num_random=300, log_mu=-3.0)
    otree = O.build(pos, idx)
    tree = gpu.upload(otree.nodes, otree.slots, pos, idx)
    full = 1 << 19
    g = torch.Generator(device="cuda").manual_seed(2)
    rays = torch.zeros((2 * full + 7, 8), device="cuda")
    rays[:, 0:3] = torch.rand((len(rays), 3), device="cuda", generator=g) * 3 - 1.5
    rays[:, 4:7] = torch.randn((len(rays), 3), device="cuda", generator=g)
    rays[:, 7] = 1e30
    want = torch.cat([tree.intersect(c.contiguous()).view(torch.int32).reshape(len(c), -1)
                      for c in rays.split(100000)])
    for n in (full + 1, 100, full, full + 1, full - 1, len(rays), 1, full + 64, len(rays)):
        print(f"{n} rays", flush=True)
        got = tree.intersect(rays[:n].contiguous()).view(torch.int32).reshape(n, -1)
        assert torch.equal(got, want[:n])


@pytest.mark.parametrize("max_bounces", [1, 4, 5])
def test_frames_after_one_another(gpu, max_bounces):
    import torch

    from sprout_amd import render, scenes

    scene = render.Scene(*scenes.room())
    cams = [render.camera(33, 17), render.camera(33, 17, fov_deg=50.0)]

    def frame(k, **kw):
        print(f"view {k} {kw}", flush=True)
        img, st = render.render(scene, cams[k], 4, 2, 1, max_bounces, seed=3, stats=True, **kw)
        torch.cuda.synchronize()
        return img.cpu().numpy(), st.extend_rays, st.shadow_rays

    want = [frame(k, graph=False) for k in (0, 1)]
    assert want[0][1] > 0 and np.isfinite(want[0][0]).all()
    # (a view seen twice running is captured and then replayed)
    for k, kw in ((0, {}), (0, {}), (0, {}), (1, {}), (0, {}), (1, dict(regenerate=True)),
                  (1, {}), (1, {}), (0, dict(regenerate=True)), (1, {})):
        img, extend, shadow = frame(k, **kw)
        assert np.array_equal(img, want[k][0])
        assert (extend, shadow) == want[k][1:]
    scene.release()
