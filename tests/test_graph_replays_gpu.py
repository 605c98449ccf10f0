"""Captured waves against a scene, an instance set or a network that changes
between frames of one view into one buffer: allocations of the same sizes
come back at the same addresses, and every frame, launched, captured or
replayed, must be the one of the scene as it is."""

import numpy as np
import pytest

from scene_util import instanced_room
from test_scene_update_gpu import lit_room, moved

pytestmark = pytest.mark.gpu

ORDER = (0, 0, 0, 1, 0, 0, 1, 1, 1, 2, 0, 1, 2, 2, 2, 0, 0)


@pytest.fixture(scope="module")
def gpu():
    import torch

    from sprout_amd import bvh, render

    assert torch.cuda.is_available(), "GPU tests need a GPU"
    bvh.init(0)
    yield render
    torch.cuda.synchronize()


def frames(change, frame):
    """frame(graph) after change(k), for k in ORDER, against the frames launched kernel by kernel"""
    want = []
    for k in range(3):
        change(k)
        want.append(frame(False))
    assert not np.array_equal(want[0], want[1]) and np.isfinite(want[0]).all()
    last = None
    for n, k in enumerate(ORDER):
        print(f"frame {n}: state {k}", flush=True)
        if k != last:
            change(k)
            last = k
        assert np.array_equal(frame(True), want[k]), (n, k)


def plain_frame(gpu, scene, **kw):
    import torch

    cam = gpu.camera(40, 30)
    acc = torch.zeros((30, 40, 3), dtype=torch.float64, device="cuda")

    def frame(graph):
        acc.zero_()
        gpu.render(scene, cam, 4, samples_per_wave=4, seed=3, graph=graph, accum=acc, **kw)
        return acc.cpu().numpy().copy()

    return frame


@pytest.mark.parametrize("regenerate", [False, True])
def test_moving_emitters(gpu, regenerate):
    pos, idx, tmat, mats = lit_room()
    rng = np.random.default_rng(7)
    # the third state crowds the small emitters together: a deeper tree
    near = moved(pos, idx, tmat, mats, 2)
    crowd = np.unique(idx[tmat == len(mats) - 1])
    near[crowd] = (near[crowd] - near[crowd].mean(0)) * 0.05 + near[crowd].mean(0)
    near += rng.uniform(-1e-4, 1e-4, near.shape).astype(np.float32)
    states = [pos, moved(pos, idx, tmat, mats, 1), near]
    scene = gpu.Scene(pos, idx, tmat, mats)
    frames(lambda k: scene.update_positions(states[k]), plain_frame(gpu, scene, regenerate=regenerate))
    scene.release()


@pytest.mark.parametrize("regenerate", [False, True])
def test_moving_instances(gpu, regenerate):
    sc = instanced_room(6, seed=4)
    states = [sc, instanced_room(6, seed=11), instanced_room(6, seed=12)]
    scene = gpu.InstancedScene(sc["meshes"], sc["mesh_of"], sc["world_to_object"], sc["object_to_world"],
                               sc["instance_materials"], sc["positions"], sc["indices"],
                               sc["triangle_materials"], sc["materials"])
    frames(lambda k: scene.update_instances(states[k]["world_to_object"], states[k]["object_to_world"]),
           plain_frame(gpu, scene, regenerate=regenerate))
    scene.release()


def test_changing_networks(gpu):
    """a network released and another made in its place"""
    import torch

    from sprout_amd import guide, scenes

    scene = gpu.Scene(*scenes.room())
    cam = gpu.camera(40, 30)
    acc = torch.zeros((30, 40, 3), dtype=torch.float64, device="cuda")
    held = []

    def change(k):
        while held:
            held.pop().release()
        held.append(guide.Guide(seed=5 + k))

    def frame(graph):
        acc.zero_()
        gpu.render_guided(scene, cam, 4, held[0], train=False, samples_per_wave=4, seed=3, graph=graph, accum=acc)
        return acc.cpu().numpy().copy()

    frames(change, frame)
    held.pop().release()
    scene.release()
