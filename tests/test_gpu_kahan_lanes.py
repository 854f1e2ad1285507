"""Compensated sums stay compensated to the end (PREC_KAHAN, per-target walk): each lane's sum
and its compensation go through the reduction over the wave and reach the store.

The terms are exact: unit-mass sources at points whose f32 squared distance from the target
(at the origin, no softening) is exactly 1, so each adds its own f32 coordinate. The f64 sum
of those is exact to 1e-13, and all are positive, so a compensated f32 sum ends within one
rounding of it, 2^-24 relative, plus the lanes' roundings of single terms: about
sqrt(n) 2^-25 of a term, below 2% of 2^-24 of the sum for n >= 500. Plain additions over 64
lanes leave up to 3 times as much."""
from __future__ import annotations

import numpy as np
import pytest

import galaxy_amd as glx

pytestmark = pytest.mark.gpu

f = np.float32


def unit_points(rng, n):
    """Points of the first octant with x^2 + y^2 + z^2 = 1 in f32, added in that order."""
    out = np.zeros((0, 3), f)
    while len(out) < n:
        v = np.abs(rng.standard_normal((4 * n, 3))) + 0.05
        v = (v / np.linalg.norm(v, axis=1, keepdims=True)).astype(f)
        r2 = (v[:, 0] * v[:, 0] + v[:, 1] * v[:, 1]) + v[:, 2] * v[:, 2]
        out = np.concatenate([out, v[r2 == f(1)]])
    return out[:n]


def system(seed, n):
    rng = np.random.default_rng(seed)
    src = unit_points(rng, n).astype(np.float64)
    # massless corners keep the centre at the origin
    pos = np.concatenate([[np.zeros(3), np.full(3, 2.0), np.full(3, -2.0)], src])
    mass = np.concatenate([[1.0, 0.0, 0.0], np.ones(n)])
    return pos, mass, src.sum(axis=0)


@pytest.mark.parametrize("build", [dict(), dict(morton_bits=63)], ids=["30", "63"])
def test_sum_is_within_one_rounding(build):
    worst = 0.0
    for seed in range(40):
        pos, mass, want = system(seed, 500 + 37 * seed)
        s = glx.Lbvh(1.0, 0.0, 1e-6, precision=glx.PREC_KAHAN, **build)
        worst = max(worst, np.abs(s.accelerations(pos, mass)[0] / want - 1.0).max())
    assert worst < 1.05 * 2.0 ** -24, worst * 2.0 ** 24


def test_group_fallback_is_the_reference_build(monkeypatch):
    """The group walk's stack-overflow fallback hands on the same compensated sums."""
    for seed in range(4):
        pos, mass, _ = system(seed, 700)
        ref = glx.Lbvh(1.0, 0.0, 1e-6, precision=glx.PREC_KAHAN).accelerations(pos, mass)
        monkeypatch.setenv("GLX_WALK_STACK_CAP", "2")
        grp = glx.Lbvh(1.0, 0.0, 1e-6, precision=glx.PREC_KAHAN, walk=glx.WALK_GROUP)
        got = grp.accelerations(pos, mass)
        monkeypatch.delenv("GLX_WALK_STACK_CAP")
        assert np.array_equal(got, ref)
