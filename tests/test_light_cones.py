"""Merging a light's cone into a tree node's (the root of two lights, one
leaf): whether the second cone lies inside the first is decided by the float
angles, whichever way the builder tells it, so lights at the very edge of a
cone are checked against angles computed here."""

import numpy as np
import pytest

from sprout_amd import lights

F = np.float32


def angle(c):
    return F(np.arccos(np.float64(F(c))))


@pytest.mark.parametrize("wide", [0.0, 1e-4, 1e-3, 0.4, 1.5, 2.5, 3.1])
@pytest.mark.parametrize("narrow", [0.0, 0.5, 1.0])
def test_a_cone_at_the_edge_of_another(wide, narrow):
    rng = np.random.default_rng(3)
    lo, hi = np.zeros((2, 3), F), np.ones((2, 3), F)
    inside = 0
    for step in [0, *np.concatenate([s * 10.0 ** np.arange(-8, -2) for s in (-1, 1)])]:
        a_angle, b_angle = wide, wide * narrow
        d = max(wide - b_angle + step, 0.0)
        x = rng.normal(size=3)
        x /= np.linalg.norm(x)
        y = np.cross(x, rng.normal(size=3))
        y /= np.linalg.norm(y)
        a = np.array([*x, np.cos(a_angle)], F)
        b = np.array([*(np.cos(d) * x + np.sin(d) * y), np.cos(b_angle)], F)
        nodes, *_ = lights.build_tree(lo, hi, np.stack([a, b]), np.ones(2, F), np.zeros(2, np.uint8))
        dot = F(F(F(a[0] * b[0]) + F(a[1] * b[1])) + F(a[2] * b[2]))
        aa, ba, da = angle(a[3]), angle(b[3]), angle(np.clip(dot, -1, 1))
        first, second = (a, b) if ba <= aa else (b, a)
        aa, ba = max(aa, ba), min(aa, ba)
        contained = np.array_equal(a, b) or min(F(da + ba), F(np.pi)) <= aa
        inside += contained
        same = np.array_equal(np.asarray(nodes["cone"][0], F), first)
        assert same or not contained
        if not contained and F(da + ba) > aa * F(1 + 1e-3) and aa < F(3):
            assert not same
    assert inside
