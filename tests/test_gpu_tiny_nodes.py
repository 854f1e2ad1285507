"""Nodes a few f32 ulps wide. A node's centre and com are rounded there, so a body inside its
box can lie farther from the com than the acceptance radius (sqrt(3) s against s / theta);
the reference rejects a node for every target inside its box. With no softening each body of
such a pair feels the other at a distance of an ulp or so, which dwarfs everything else: an
accepted pair would add the body's own mass and double the force."""
from __future__ import annotations

import numpy as np
import pytest

import galaxy_amd as glx
from tests import inputs as I

pytestmark = pytest.mark.gpu

THETAS = [0.5, 0.6, 0.7, 0.9, 1.0, 1.3]
BUILDS = {
    "reference": dict(),
    "reference63": dict(morton_bits=63),
    "kahan": dict(precision=glx.PREC_KAHAN),
    "abs32": dict(precision=glx.PREC_ABS32),
}


def check(pos, mass, rows, theta, **build):
    acc = glx.Lbvh(1.0, 0.0, theta, **build).accelerations(pos, mass)[rows]
    ref = glx.direct_sum_f64(pos, mass, 1.0, 0.0, rows)
    # positions are exact in f32, so a pair's term is good to a few ulps; all other terms
    # together are below 1e-6 of it
    err = np.linalg.norm(acc - ref, axis=1) / np.linalg.norm(ref, axis=1)
    assert err.max() < 1e-5, (err.max(), int((err > 1e-5).sum()))


@pytest.mark.parametrize("theta", THETAS)
@pytest.mark.parametrize("build", sorted(BUILDS))
def test_pair_one_ulp_apart(theta, build):
    a = np.full(3, 0.75)
    b = a + 2.0 ** -24
    pos = np.array([a, b, -b])
    check(pos, np.ones(3), np.array([0, 1]), theta, **BUILDS[build])
    pos = np.concatenate([[np.full(3, 1.0), np.full(3, 1.0 + 2.0 ** -23)],
                          np.full((1, 3), 8.0), np.full((1, 3), -8.0)])
    check(pos, np.ones(4), np.array([0, 1]), theta, **BUILDS[build])


def ulp_pairs(rng, pairs, most):
    """Pairs up to `most` ulps apart on each axis, exact in f32 about a centre at 0."""
    a = rng.uniform(0.26, 0.99, (pairs, 3)).astype(np.float32)
    a *= np.where(rng.random((pairs, 3)) < 0.5, -1, 1).astype(np.float32)
    step = rng.integers(0, most + 1, (pairs, 3)).astype(np.float64)
    step[step.sum(axis=1) == 0] = 1.0
    b = (a + step * np.spacing(np.abs(a))).astype(np.float32)
    pos = np.concatenate([np.stack([a, b], 1).reshape(-1, 3), [[1.0] * 3, [-1.0] * 3]])
    return pos.astype(np.float64), 2 * pairs


@pytest.mark.parametrize("theta", THETAS)
@pytest.mark.parametrize("build", sorted(BUILDS))
def test_random_pairs_up_to_three_ulps(theta, build):
    rng = np.random.default_rng(11)
    pos, k = ulp_pairs(rng, 400, 3)
    mass = rng.uniform(0.5, 1.5, len(pos))
    check(pos, mass, np.arange(k), theta, **BUILDS[build])
