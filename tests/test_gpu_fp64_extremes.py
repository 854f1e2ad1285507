"""FP64 direct sum and potential where the fast forms of a term do not apply: a body's own
term is left out whatever its mass, and separations whose square is not a normal f32."""
from __future__ import annotations

import numpy as np
import pytest

import galaxy_amd as glx

pytestmark = pytest.mark.gpu


def rows(pos, mass, g, eps, targets):
    """The sum in f64, each target left out of its own row."""
    out = np.zeros((len(targets), 3))
    for q, t in enumerate(targets):
        d = np.delete(pos, t, 0) - pos[t]
        r2 = (d * d).sum(1) + eps * eps
        out[q] = g * (np.delete(mass, t)[:, None] * d / (r2 * np.sqrt(r2))[:, None]).sum(0)
    return out


# n and targets: one chunk, several chunks, a block of targets that straddles chunks
@pytest.mark.parametrize("n", [3, 130, 5003])
@pytest.mark.parametrize("own", [np.inf, -np.inf, np.nan, 1e300])
@pytest.mark.parametrize("eps", [0.0, 1e-20, 0.05])
def test_own_mass_is_left_out(n, own, eps):
    rng = np.random.default_rng(n)
    pos = rng.standard_normal((n, 3))
    mass = rng.uniform(0.5, 1.5, n)
    t = n // 2
    mass[t] = own
    got = glx.direct_sum_f64(pos, mass, 1.0, eps, np.array([t]))
    with np.errstate(all="ignore"):
        ref = rows(pos, mass, 1.0, eps, [t])
    assert np.isfinite(got).all()
    assert np.abs(got - ref).max() < 1e-12 * np.abs(ref).max()


def test_own_mass_among_other_targets():
    rng = np.random.default_rng(5)
    n = 5003
    pos = rng.standard_normal((n, 3))
    mass = rng.uniform(0.5, 1.5, n)
    mass[77] = np.inf
    tgt = np.arange(0, n, 7)  # 77 is one of them
    got = glx.direct_sum_f64(pos, mass, 1.0, 0.05, tgt)
    ref = rows(pos, mass, 1.0, 0.05, [77])[0]
    q = int(np.where(tgt == 77)[0][0])
    assert np.abs(got[q] - ref).max() < 1e-12 * np.abs(ref).max()
    assert not np.isfinite(np.delete(got, q, 0)).any()  # every other row holds the infinity


@pytest.mark.parametrize("n", [2, 65, 200, 3000])
@pytest.mark.parametrize("at", ["first", "inside"])
def test_potential_with_an_infinite_mass(n, at):
    """Only the pairs j > i count: an infinite mass makes the energy -inf, not NaN."""
    rng = np.random.default_rng(n)
    pos = rng.standard_normal((n, 3))
    mass = rng.uniform(0.5, 1.5, n)
    mass[0 if at == "first" else (n - 1) // 2] = np.inf
    assert glx.Lbvh(1.0, 0.05, 0.5).potential_energy(pos, mass) == -np.inf


# squared separations from below the smallest f32 to above the largest
@pytest.mark.parametrize("scale", [1e-24, 1e-22, 1e-21, 3e-21, 1e-20, 3e-20, 1e-19, 1e-18,
                                   1e18, 1.5e19, 1e20])
def test_separations_beyond_normal_f32(scale):
    rng = np.random.default_rng(3)
    n = 70
    pos = scale * rng.standard_normal((n, 3))
    mass = rng.uniform(0.5, 1.5, n)
    tgt = np.arange(n)
    got = glx.direct_sum_f64(pos, mass, 1.0, 0.0, tgt)
    ref = rows(pos, mass, 1.0, 0.0, tgt)
    assert np.abs(got - ref).max() < 1e-13 * np.abs(ref).max()
    i, j = np.triu_indices(n, 1)
    pot = -(mass[i] * mass[j] / np.linalg.norm(pos[i] - pos[j], axis=1)).sum()
    u = glx.Lbvh(1.0, 0.0, 0.5).potential_energy(pos, mass)
    assert abs(u / pot - 1.0) < 1e-13
