"""The default traversal over the launch sizes and ray forms where its rules
change: slices of fewer than 64 rays a wave, the last slice, the first
claimed ray; rays with zero, NaN or infinite components, and rays that start
on a node's bound with an infinite inverse direction there, also through
instances; trees whose bounds are not finite.  Every word must equal the reference-order loop's
(mi_trace_counts), which the other tests pin to the oracle."""

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


@pytest.fixture(scope="module")
def mesh():
    from sprout_amd import scenes

    pos, idx = scenes.displaced_icosphere(subdivisions=3, num_random=700, log_mu=-3.0)
    return pos, idx, O.build(pos, idx)


def rays_of(n, seed=1):
    rng = np.random.default_rng(seed)
    r = np.zeros((n, 8), np.float32)
    r[:, 0:3] = rng.uniform(-1.5, 1.5, (n, 3))
    r[:, 4:7] = rng.normal(size=(n, 3))
    r[:, 7] = 3.4028235e38
    return r


def agree(gpu, tree, rays, kernels=(3, 4)):
    import torch

    d = torch.from_numpy(rays).cuda()
    for any_hit in (False, True):
        want, _ = tree.counts(d, any_hit=any_hit)
        for kernel in kernels:
            gpu.set_trace_config(kernel=kernel)
            got = tree.intersect_p(d) if any_hit else tree.intersect(d)
            torch.cuda.synchronize()
            gpu.set_trace_config(kernel=3)
            assert torch.equal(got, want), (kernel, any_hit)
    return want


# one ray a wave up to 16 waves per CU (4096), the 64-ray slices of 2^18
# rays on either side, claimed rays past the resident grid's 2^19
@pytest.mark.parametrize("n", [1, 2, 63, 64, 65, 4095, 4097, 8193, 262143, 262145, 524289, 700001])
def test_launch_sizes(gpu, mesh, n):
    pos, idx, otree = mesh
    print(f"{n} rays", flush=True)
    tree = gpu.upload(otree.nodes, otree.slots, pos, idx)
    occluded = agree(gpu, tree, rays_of(n))
    if n > 1000:
        assert 0 < int(occluded.sum()) < n


@pytest.mark.parametrize("shape", [(64, 1), (256, 1), (1024, 1), (64, 8)])
def test_small_grids_claim_the_rest(gpu, mesh, shape):
    """few waves: most rays come from the claim counters"""
    import torch

    pos, idx, otree = mesh
    tree = gpu.upload(otree.nodes, otree.slots, pos, idx)
    d = torch.from_numpy(rays_of(300007)).cuda()
    want, _ = tree.counts(d)
    gpu.set_trace_config(block_size=shape[0], blocks_per_cu=shape[1], lds_entries=3, claim_batch=7)
    got = tree.intersect(d)
    torch.cuda.synchronize()
    gpu.set_trace_config()
    assert torch.equal(got, want)


def test_odd_ray_forms(gpu, mesh):
    pos, idx, otree = mesh
    tree = gpu.upload(otree.nodes, otree.slots, pos, idx)
    r = rays_of(4096, 2)
    special = np.array([0.0, -0.0, np.inf, -np.inf, np.nan, 1e-42, -1e-42, 3e38, 1e-30], np.float32)
    rng = np.random.default_rng(3)
    for i in range(len(r)):
        for c in rng.choice(8, rng.integers(0, 4), replace=False):
            r[i, c] = special[rng.integers(len(special))]
    r[0, 4:7] = 0.0            # no direction at all
    r[1, 4:7] = np.nan
    r[2, 4:7] = (0, 0, 1)      # along an axis
    r[3, 4:7] = (0, -0.0, -1)
    r[4, 3], r[4, 7] = 2.0, 1.0  # an empty interval
    agree(gpu, tree, r)


@pytest.mark.parametrize("value", [np.nan, np.inf, -np.inf])
def test_bounds_not_finite(gpu, mesh, value):
    """an uploaded tree whose bounds are not finite in places"""
    pos, idx, otree = mesh
    nodes = otree.nodes.copy()
    rng = np.random.default_rng(4)
    pick = rng.choice(len(nodes), len(nodes) // 8, replace=False)
    nodes["lo" if value < 0 or np.isnan(value) else "hi"][pick, rng.integers(0, 3, len(pick))] = value
    tree = gpu.upload(nodes, otree.slots, pos, idx)
    agree(gpu, tree, rays_of(4096, 5))


def test_vertex_not_finite(gpu, mesh):
    """a built tree over a mesh with a NaN coordinate"""
    import torch

    pos, idx, _ = mesh
    p = pos.copy()
    p[7, 1] = np.nan
    tree = gpu.Builder_SAH().build(torch.from_numpy(p).cuda(),
                                   torch.from_numpy(idx.view(np.int32)).cuda())
    agree(gpu, tree, rays_of(4096, 6))


@pytest.mark.parametrize("value", [np.nan, np.inf, -np.inf])
def test_hits_beside_a_vertex_not_finite(gpu, mesh, value):
    """the other triangles of such a mesh are hit as if it were not there,
    alone and instanced"""
    import torch

    from sprout_amd import instances

    pos, idx, _ = mesh
    p = pos.copy()
    p[7, 1] = p[300, 0] = value
    tree = gpu.Builder_SAH().build(torch.from_numpy(p).cuda(),
                                   torch.from_numpy(idx.view(np.int32)).cuda())
    rays = rays_of(4096, 8)
    d = torch.from_numpy(rays).cuda()
    bad = ~np.isfinite(p[idx].reshape(len(idx), -1)).all(axis=1)
    q = p.copy()
    q[~np.isfinite(q)] = 0.0
    want = O.brute_force(q, idx[~bad], rays)
    ids = np.flatnonzero(~bad).astype(np.uint32)
    hit = want[:, 3] != 0xFFFFFFFF
    want[hit, 3] = ids[want[hit, 3]]
    assert bad.any() and hit.mean() > 0.25
    for kernel in (2, 3, 4):
        gpu.set_trace_config(kernel=kernel)
        got = tree.intersect(d).cpu().numpy().view(np.uint32)
        gpu.set_trace_config(kernel=3)
        assert np.array_equal(got, want), kernel
    eye = np.eye(4, dtype=np.float32)[None]
    inst = instances.Instances([tree], eye, eye)
    got = inst.intersect(d).cpu().numpy().view(np.uint32)
    assert np.array_equal(got[:, :4], want)
    inst.release()


def rays_on_planes(n, seed, values):
    """rays along the planes x, y or z = one of values (and edges, where two
    axes are chosen), with direction components there whose inverse is
    infinite (1e-20, 1e-30, 3.7e-33, 5.4e-20), zero's NaN or finite"""
    r = rays_of(n, seed)
    rng = np.random.default_rng(seed + 1)
    flat = np.array([1e-20, -1e-20, 1e-30, -1e-30, 3.7e-33, -3.7e-33, 5.4e-20, -5.4e-20, 0.0, 6e-17], np.float32)
    for i in range(n):
        for c in rng.choice(3, rng.integers(1, 3), replace=False):
            v = values[c]
            r[i, c] = v[rng.integers(len(v))]
            r[i, 4 + c] = flat[rng.integers(len(flat))]
    return r


def grid_mesh(n):
    """a flat n x n grid at z = 0 whose lines are bounds of its nodes"""
    x, y = np.meshgrid(np.arange(n + 1), np.arange(n + 1), indexing="ij")
    pos = np.stack([x, y, 0.25 * ((x + y) % 2)], -1).reshape(-1, 3).astype(np.float32) / n - np.float32(0.5)
    a = (np.arange(n)[:, None] * (n + 1) + np.arange(n)[None, :]).reshape(-1)
    idx = np.concatenate([np.stack([a, a + n + 1, a + n + 2], 1), np.stack([a, a + n + 2, a + 1], 1)])
    return pos, idx.astype(np.uint32)


@pytest.mark.parametrize("which", ["grid", "sphere"])
def test_origins_on_bounds(gpu, mesh, which):
    pos, idx, otree = mesh
    if which == "grid":
        pos, idx = grid_mesh(16)
        otree = O.build(pos, idx)
    tree = gpu.upload(otree.nodes, otree.slots, pos, idx)
    planes = [np.concatenate([otree.nodes["lo"][:, c], otree.nodes["hi"][:, c]]) for c in range(3)]
    rays = rays_on_planes(20000, 11, planes)
    agree(gpu, tree, rays, kernels=(2, 3))
    # and against the oracle's own walk
    import torch

    d = torch.from_numpy(rays).cuda()
    got = tree.intersect(d).cpu().numpy().view(np.uint32)
    want = O.trace(otree, pos, idx, rays)
    assert np.array_equal(got, want)
    assert (want[:, 3] != 0xFFFFFFFF).mean() > 0.05
    # the compressed boxes of kernel 4 are larger: it may also find a hit in a
    # box that a ray along its plane misses by a rounding, and loses none
    gpu.set_trace_config(kernel=4)
    wide = tree.intersect(d).cpu().numpy().view(np.uint32)
    gpu.set_trace_config(kernel=3)
    more = np.any(wide != want, axis=1)
    nearest = O.brute_force(pos, idx, rays)
    assert (wide[more, 0].view(np.float32) <= want[more, 0].view(np.float32)).all()
    assert (wide[more, 0].view(np.float32) >= nearest[more, 0].view(np.float32)).all()
    assert more.mean() < 0.05


def test_origins_on_bounds_of_instances(gpu):
    """the instances are moved by whole grid cells, so that a world ray on a
    plane of the grid is on one in object space too"""
    import torch

    from sprout_amd import instances

    pos, idx = grid_mesh(8)
    tree = gpu.Builder_SAH().build(torch.from_numpy(pos).cuda(), torch.from_numpy(idx.view(np.int32)).cuda())
    n = 9
    o2w = np.tile(np.eye(4, dtype=np.float32), (n, 1, 1))
    o2w[:, 3, :3] = [(i % 3 - 1, i // 3 - 1, 0.25 * (i % 2)) for i in range(n)]
    w2o = np.linalg.inv(o2w.astype(np.float64)).astype(np.float32)
    inst = instances.Instances([tree] * n, w2o, o2w)
    ref = O.Instances([(pos, idx, O.build(pos, idx))], np.zeros(n, np.uint32), w2o, o2w)
    lines = [np.arange(-12, 13, dtype=np.float32) / 8] * 2 + [np.arange(-4, 5, dtype=np.float32) / 8]
    rays = rays_on_planes(20000, 21, lines)
    d = torch.from_numpy(rays).cuda()
    for any_hit in (False, True):
        got = (inst.intersect_p(d) if any_hit else inst.intersect(d)).cpu().numpy().view(np.uint32)
        want = ref.trace(rays, any_hit=any_hit)
        assert np.array_equal(got if any_hit else got[:, :5], want), any_hit
    assert want.mean() > 0.05
    inst.release()


def test_captured_launch_after_a_smaller_one(gpu, mesh):
    """a captured launch's stack area stays its own when a smaller launch,
    with more waves, follows: replays give the same hits"""
    import torch

    pos, idx, otree = mesh
    tree = gpu.upload(otree.nodes, otree.slots, pos, idx)
    gpu.set_trace_config(lds_entries=1)  # every walk spills
    d = torch.from_numpy(rays_of(5000, 31)).cuda()
    small = d[:4000].contiguous()
    want = tree.intersect(d).clone()  # reserves
    hits = torch.empty_like(want)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        tree.intersect(d, hits)
    with torch.cuda.graph(torch.cuda.CUDAGraph()):
        tree.intersect(small)  # nothing is allocated inside a capture
    for _ in range(3):
        assert torch.equal(tree.intersect(small), want[:4000])
        hits.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(hits, want)
    gpu.set_trace_config()
    assert torch.equal(tree.counts(d)[0], want)
