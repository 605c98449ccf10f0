"""The default traversal over the launch sizes and ray forms where its rules
change: slices of fewer than 64 rays a wave, the last slice, the first
claimed ray; rays with zero, NaN or infinite components; trees whose bounds
are not finite.  Every word must equal the reference-order loop's
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


def agree(gpu, tree, rays):
    import torch

    d = torch.from_numpy(rays).cuda()
    for any_hit in (False, True):
        want, _ = tree.counts(d, any_hit=any_hit)
        for kernel in (3, 4):
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
