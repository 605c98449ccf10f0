"""The device light-tree builder at the sizes where its kernels change path,
against the host builder byte for byte: a wave folds 64 lights at a time (63
to 65, and last chunks whose powers end inside a group of eight), the split's
workgroup takes 256 candidates (85 and 86 lights: 255 and 258) and 256 lights
(255 to 257, 513) a pass, sweep and grid (127, 128), lights in one plane
(infinite costs), duplicated lights (equal costs), lights without power, and
a tree deep enough that its levels' bounds start over (64)."""

import numpy as np
import pytest

from sprout_amd import lights

pytestmark = pytest.mark.gpu

F = np.float32


@pytest.fixture(scope="module")
def gpu():
    import torch

    from sprout_amd import bvh

    assert torch.cuda.is_available(), "GPU tests need a GPU"
    bvh.init(0)
    yield
    torch.cuda.synchronize()


def make(n, form, seed):
    rng = np.random.default_rng(seed)
    c = rng.uniform(-2, 2, (n, 3)).astype(F)
    if form == "plane":
        c[:, 2] = F(0.5)
    if form == "twins":
        c[1::2] = c[: len(c[1::2]) * 2 : 2]
    if form == "deep":  # every split cuts off the far light: one level a light
        c[:] = F(0)
        c[:, 0] = (1e-6 * 1.7 ** np.arange(n)).astype(F)
    e = rng.uniform(0.01, 0.2, (n, 3)).astype(F)
    if form == "plane":
        e[:, 2] = 0
    if form == "twins":
        e[:] = F(0.05)
    if form == "deep":
        e = np.repeat(c[:, :1], 3, 1) * F(1e-8)
    nrm = rng.normal(size=(n, 3))
    nrm /= np.linalg.norm(nrm, axis=1, keepdims=True)
    cones = np.concatenate([nrm, rng.uniform(0.2, 1.0, (n, 1))], 1).astype(F)
    powers = np.exp(rng.normal(size=n)).astype(F)
    if form == "deep":
        cones[:] = cones[0]
        powers[:] = F(1e-8)
    if form == "dark":
        powers[::9] = 0
    return (c - e).astype(F), (c + e).astype(F), cones, powers, (rng.random(n) < (0 if form == "deep" else 0.3)).astype(np.uint8)


def same(host, dev):
    for a, b in zip(host, dev):
        a, b = np.asarray(a), np.asarray(b)
        assert a.tobytes() == b.tobytes()


def depth(nodes):
    bits = np.asarray(nodes).view(np.uint32).reshape(len(nodes), -1)[:, 10]
    deep, todo = 0, [(0, 0)]
    while todo:
        i, d = todo.pop()
        deep = max(deep, d)
        if bits[i] & 1:
            todo += [(int(bits[i] >> 2), d + 1), (int(bits[i] >> 2) + 1, d + 1)]
    return deep


@pytest.mark.parametrize("n", [4, 5, 63, 64, 65, 85, 86, 127, 128, 255, 256, 257, 513])
@pytest.mark.parametrize("form", ["any", "plane", "twins", "dark"])
def test_scene_tree_at_its_edges(gpu, n, form):
    lights_in = make(n, form, 100 + n)
    print(f"{n} lights, {form}", flush=True)
    same(lights.build_tree(*lights_in), lights.build_tree_device(*lights_in))


def test_a_deep_tree(gpu):
    lights_in = make(127, "deep", 7)
    host = lights.build_tree(*lights_in)
    print(f"depth {depth(host[0])}", flush=True)
    assert depth(host[0]) > 64
    same(host, lights.build_tree_device(*lights_in))


def test_parts_at_their_edges(gpu):
    sizes = [1, 64, 65, 4, 31, 32, 255, 256, 257, 321]
    parts = [make(s, "dark" if k % 2 else "any", 200 + k) for k, s in enumerate(sizes)]
    first = np.concatenate([[0], np.cumsum(sizes)]).astype(np.uint32)
    lo, hi, cones, powers = (np.concatenate([p[k] for p in parts]) for k in range(4))
    part_cones = np.array([[0, 0, 1, 0.3]] * len(sizes), F)
    dev = lights.build_part_trees_device(lo, hi, cones, powers, first, part_cones)
    for k in range(len(sizes)):
        b, e = first[k], first[k + 1]
        print(f"part of {sizes[k]} lights", flush=True)
        same(lights.build_part_tree(lo[b:e], hi[b:e], cones[b:e], powers[b:e], part_cones[k]), dev[k])
