"""A massless body at a NaN position takes part in no force: the other bodies' rows are those
of the direct sum without it, in the reference build and in the group walk's, wherever it
sorts (one NaN axis, all three) and however few bodies there are. The com of every node
above it is NaN; such nodes are opened and the body's own leaf is skipped."""
from __future__ import annotations

import numpy as np
import pytest

import galaxy_amd as glx
from oracle import oracle as O
from tests import inputs as I

pytestmark = pytest.mark.gpu

BUILDS = {
    "reference": dict(),
    "kahan": dict(precision=glx.PREC_KAHAN),
    "reference63": dict(morton_bits=63),
    "counted": dict(count=True),
    "group": dict(morton_bits=63, walk=glx.WALK_GROUP, multipole=2),
}


@pytest.mark.parametrize("n", [1, 2, 3, 5, 64, 300])
@pytest.mark.parametrize("axes", [(0,), (2,), (0, 1, 2)])
@pytest.mark.parametrize("build", sorted(BUILDS))
def test_massless_nan_body_pulls_nobody(n, axes, build):
    pos, _, mass = I.cluster(n, n)
    at = n // 2
    p = np.insert(pos, at, 0.25, axis=0)
    p[at, list(axes)] = np.nan
    m = np.insert(mass, at, 0.0)
    acc = glx.Lbvh(1.0, 0.05, 1e-6, **BUILDS[build]).accelerations(p, m)
    got = np.delete(acc, at, axis=0)
    assert np.isfinite(got).all()
    ref = O.direct_sum(pos, mass, 1.0, 0.05)
    if n == 1:
        assert np.array_equal(got, ref)
    else:
        assert I.rms_rel_err(got, ref) < 2e-5  # the f32 walk's measure at theta -> 0


def test_lone_nan_body():
    """No other body: nothing is summed, so the row is 0."""
    acc = glx.Lbvh(1.0, 0.05, 0.5).accelerations(np.full((1, 3), np.nan), np.ones(1))
    assert np.array_equal(acc, np.zeros((1, 3)))
