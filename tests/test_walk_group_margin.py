"""The group walk's acceptance for theta <= 1 (galaxy_amd/csrc/glx_kernels.hip, walk_group_box and
walk_round, near_share) on its f32 arithmetic, for nodes down to an ulp wide at the edge of group boxes up
to 1e6 times larger: a node that holds a body within the group box is never accepted, unless
it is a single point. The acceptance radius alone would let many through."""
from __future__ import annotations

import numpy as np

f = np.float32


def norm2(e):
    return ((e[:, 0] * e[:, 0] + e[:, 1] * e[:, 1]) + e[:, 2] * e[:, 2]).astype(f)


def cases(rng, n):
    lo = (10.0 ** rng.uniform(-3, 2.9, (n, 3))).astype(f)
    lo *= np.where(rng.random((n, 3)) < 0.2, f(-1), f(1))
    hi = (lo + 10.0 ** rng.uniform(-4, 3, (n, 3))).astype(f)
    # the node: from a body at a corner of the group box, a few ulps or a small size wide
    corner = np.where(rng.random((n, 3)) < 0.5, lo, hi)
    width = np.where(rng.random((n, 1)) < 0.5, rng.integers(0, 60, (n, 3)) * np.spacing(np.abs(corner)),
                     10.0 ** rng.uniform(-8, -3, (n, 1)) * rng.random((n, 3)))
    other = (corner + width * np.where(rng.random((n, 3)) < 0.5, -1, 1)).astype(f)
    mn, mx = np.minimum(corner, other), np.maximum(corner, other)
    com = np.clip((mn + rng.random((n, 3)).astype(f) * (mx - mn)).astype(f), mn, mx)
    ends = rng.random(n) < 0.5
    com[ends] = np.where(rng.random((int(ends.sum()), 3)) < 0.5, mn[ends], mx[ends])
    return lo, hi, mn, mx, com


def test_no_node_with_a_body_in_the_group_is_accepted():
    rng = np.random.default_rng(4)
    by_radius = 0
    for theta in (0.05, 0.3, 0.5, 0.7, 0.9, 1.0):
        for _ in range(4):
            lo, hi, mn, mx, com = cases(rng, 100_000)
            cen, half = ((mn + mx) * f(0.5)).astype(f), ((mx - mn) * f(0.5)).astype(f)
            size = (f(2) * half.max(axis=1)).astype(f)
            delta = np.sqrt(norm2((com - cen).astype(f))).astype(f)
            r = (size * f(f(1) / f(theta)) + delta).astype(f)
            gc, gh = (f(0.5) * (lo + hi)).astype(f), (f(0.5) * (hi - lo)).astype(f)
            e = np.maximum(np.abs((com - gc).astype(f)) - gh, f(0)).astype(f)
            dmin2 = norm2(e)
            accept = (dmin2 >= (r * r).astype(f)) & (size > 0)
            by_radius += int(accept.sum())
            most = np.maximum(np.abs(lo), np.abs(hi)).max(axis=1)
            share = f((24 + 20 * theta / (1 - 0.866 * theta)) * 2.0 ** -24)
            t = (most * share).astype(f)
            assert not (accept & (dmin2 >= t * t)).any(), theta
    assert by_radius > 10_000
