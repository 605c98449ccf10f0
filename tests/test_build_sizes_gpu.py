"""The builder at the sizes where a node changes list (a wave's node of 64
references, a workgroup's of 1024, more than one chunk) and at the settings
that move those lines, node for node against the oracle."""

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


def soup(n, seed, long=0.1):
    """n triangles, a tenth of them long ones that straddle many planes"""
    rng = np.random.default_rng(seed)
    c = rng.random((n, 1, 3))
    size = np.where(rng.random((n, 1, 1)) < long, 0.6, 0.05)
    pos = (c + size * (rng.random((n, 3, 3)) - 0.5)).astype(np.float32).reshape(-1, 3)
    return pos, np.arange(3 * n, dtype=np.uint32).reshape(-1, 3)


def check(gpu, pos, idx, **settings):
    import torch

    tree = gpu.Builder_SAH(**settings).build(torch.from_numpy(pos).cuda(),
                                             torch.from_numpy(idx.view(np.int32)).cuda())
    nodes, slots = tree.download()
    want = O.build(pos, idx, **settings)
    assert O.nodes_equal(nodes.view(O.NODE_DTYPE), want.nodes)
    assert np.array_equal(slots, want.slots)
    return tree


@pytest.mark.parametrize("n", [1, 4, 5, 63, 64, 65, 255, 1023, 1024, 1025, 2047, 2049, 4100, 30011])
def test_sizes(gpu, n):
    print(f"{n} triangles", flush=True)
    check(gpu, *soup(n, n))


@pytest.mark.parametrize("settings", [
    dict(num_slices=64), dict(num_slices=1), dict(sweep_threshold=1024), dict(sweep_threshold=200),
    dict(sweep_threshold=1), dict(max_primitives=1), dict(max_primitives=40),
    dict(max_primitives=100, sweep_threshold=64), dict(sweep_threshold=3, max_primitives=8)])
@pytest.mark.parametrize("n", [1500, 6000])
def test_settings(gpu, settings, n):
    print(f"{n} triangles, {settings}", flush=True)
    check(gpu, *soup(n, 7), **settings)


@pytest.mark.parametrize("level", [0, 1])
def test_the_level_of_an_unsplittable_node(gpu, level):
    """300 times one triangle, alone or beside a soup that the root splits off"""
    import torch

    from sprout_amd import _lib

    one = np.array([[0, 0, 0], [0.1, 0, 0], [0, 0.1, 0.1]], np.float32)
    pos = np.tile(one, (300, 1))
    if level:
        pos = np.concatenate([pos, soup(600, 5)[0] + np.float32(50)])
    idx = np.arange(len(pos), dtype=np.int32).reshape(-1, 3)
    with pytest.raises(_lib.MiError, match=rf"cannot be split \(level {level}\)"):
        gpu.Builder_SAH().build(torch.from_numpy(pos).cuda(), torch.from_numpy(idx).cuda())


def coordinates_not_finite(pos, value, triangles):
    """value at a corner of each of the triangles of a soup, all three
    corners on one axis for the last; and the soup whose boxes are those of
    the finite coordinates"""
    p = pos.reshape(-1, 3, 3).copy()
    rng = np.random.default_rng(len(p))
    at = rng.choice(len(p), triangles, replace=False)
    for t in at[:-1]:
        p[t, rng.integers(3), rng.integers(3)] = value
    p[at[-1], :, 1] = value
    q = p.copy()
    for t in at:
        for k in range(3):
            ok = np.isfinite(p[t, :, k])
            q[t, ~ok, k] = p[t, ok, k][0] if ok.any() else 0.0
    return p.reshape(-1, 3), q.reshape(-1, 3)


@pytest.mark.parametrize("value", [0x7FC00000, 0xFFC00000, 0x7F800000, 0xFF800000])
@pytest.mark.parametrize("n", [1, 4, 20, 21, 64, 80, 1100, 5000])
def test_vertices_not_finite(gpu, value, n):
    """the tree of the finite coordinates, whatever the others' signs"""
    import torch

    print(f"{n} triangles, {value:08x}", flush=True)
    pos, idx = soup(n, 3 * n)
    p, q = coordinates_not_finite(pos, np.uint32(value).view(np.float32), min(n, 9))
    tree = gpu.Builder_SAH().build(torch.from_numpy(p).cuda(), torch.from_numpy(idx.view(np.int32)).cuda())
    nodes, slots = tree.download()
    want = O.build(q, idx)
    assert O.nodes_equal(nodes.view(O.NODE_DTYPE), want.nodes)
    assert np.array_equal(slots, want.slots)


def test_more_references_than_a_quarter_over(gpu):
    """a fifth of the triangles long: the levels outgrow the first two allocations"""
    pos, idx = soup(20000, 9, long=0.2)
    tree = check(gpu, pos, idx)
    assert tree.info().num_slots > 2.6 * len(idx)
