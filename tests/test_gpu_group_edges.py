"""Close pairs at the edge of their walk group's box. The group walk measures a node's distance
from the group box by the box's centre and half extent, which are rounded; a pair much closer
than that rounding must still be opened by its own group, not accepted with the bodies' own
masses in it. With no softening a pair's force dwarfs everything else, so an accepted pair
shows as a wrong force."""
from __future__ import annotations

import numpy as np
import pytest

import galaxy_amd as glx

pytestmark = pytest.mark.gpu

BUILDS = {
    "monopole": dict(multipole=0),
    "quadrupole": dict(multipole=2),
    "far": dict(multipole=2, far_theta=0.6, mono_ratio=0.9),
    "buckets": dict(multipole=2, leaf_size=2),
    "abs32": dict(multipole=2, precision=glx.PREC_ABS32),
}


def system(rng):
    """Dense clumps in seven octants, so that the eighth's few bodies are one group, whose
    lowest corner is a pair a few ulps wide."""
    sign = np.array([[x, y, z] for x in (-1, 1) for y in (-1, 1) for z in (-1, 1)][:-1], float)
    clump = np.repeat(sign, 80, axis=0) * 500.0 + rng.uniform(-1, 1, (560, 3))
    low = 10.0 ** rng.uniform(-3, 1, 3)
    spread = low + rng.uniform(5, 900, (12, 3))
    a = low.astype(np.float32)
    b = (a + rng.integers(0, 40, 3) * np.spacing(a)).astype(np.float32)
    b[0] = np.nextafter(b[0], np.float32(np.inf))
    pos = np.concatenate([clump, spread, [a, b], [[1024.0] * 3, [-1024.0] * 3]])
    return pos.astype(np.float32).astype(np.float64), np.array([572, 573])


@pytest.mark.parametrize("theta", [0.4, 0.5, 0.7, 1.0, 1.3])
@pytest.mark.parametrize("build", sorted(BUILDS))
def test_pair_at_the_edge_of_its_group(build, theta):
    rng = np.random.default_rng(2)
    worst = 0.0
    for _ in range(60):
        pos, rows = system(rng)
        mass = rng.uniform(0.5, 1.5, len(pos))
        s = glx.Lbvh(1.0, 0.0, theta, morton_bits=63, walk=glx.WALK_GROUP, **BUILDS[build])
        acc = s.accelerations(pos, mass)[rows]
        ref = glx.direct_sum_f64(pos, mass, 1.0, 0.0, rows)
        err = np.linalg.norm(acc - ref, axis=1) / np.linalg.norm(ref, axis=1)
        worst = max(worst, err.max())
    assert worst < 1e-4, worst  # f32 terms; all other bodies together are below 1e-5 of a pair
