"""The per-target walk reads a node's box only for accepted distances up to the record's corner
distance (galaxy_amd/csrc/glx_kernels.hip, store_node and target_walk). On their f32 arithmetic:
a target in the box never has a greater squared distance from the com, whatever the box's size
in ulps and wherever the com is, one rounded out of its box included."""
from __future__ import annotations

import numpy as np

f = np.float32


def sq(d):
    return ((d[:, 0] * d[:, 0] + d[:, 1] * d[:, 1]) + d[:, 2] * d[:, 2]).astype(f)


def boxes(rng, n):
    a = (rng.standard_normal((n, 3)) * rng.choice([1e-3, 1.0, 1e4])).astype(f)
    kind = rng.integers(0, 3)
    if kind == 0:  # a few ulps wide
        b = (a + rng.integers(0, 5, (n, 3)) * np.spacing(np.abs(a))).astype(f)
    else:
        b = (a + rng.random((n, 3)) ** 4 * rng.choice([1e-4, 1.0, 50.0])).astype(f)
    mn, mx = np.minimum(a, b), np.maximum(a, b)
    com = (mn + rng.random((n, 3)).astype(f) * (mx - mn)).astype(f)
    out = rng.random(n) < 0.3
    com[out] += (rng.integers(-2, 3, (int(out.sum()), 3)) *
                 np.spacing(np.abs(com[out]))).astype(f)
    return mn, mx, com


def test_no_target_in_the_box_is_beyond_the_corner_distance():
    rng = np.random.default_rng(3)
    beyond_radius = 0
    for _ in range(30):
        mn, mx, com = boxes(rng, 40_000)
        e = np.maximum((com - mn).astype(f), (mx - com).astype(f))
        corner2 = sq(e)
        x = (mn + rng.random(mn.shape).astype(f) * (mx - mn)).astype(f)
        x = np.clip(x, mn, mx)
        at = rng.random(mn.shape)
        x = np.where(at < 0.3, mn, np.where(at < 0.6, mx, x))
        d2 = sq((com - x).astype(f))
        assert (d2 <= corner2).all()
        # ... while the acceptance radius at theta = 1 alone would let some of them through
        cen, half = ((mn + mx) * f(0.5)).astype(f), ((mx - mn) * f(0.5)).astype(f)
        r = (f(2) * half.max(axis=1) + np.sqrt(sq((com - cen).astype(f)))).astype(f)
        beyond_radius += int((d2 >= r * r).sum())
    assert beyond_radius > 0
