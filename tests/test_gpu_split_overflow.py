"""Stack overflow in the group walk's split form (small launches that do not count): the
producer marks the round, the other waves leave the ring, the draining wave walks the group
per target on the shared stack, and the next group takes the LDS over.

* Every group overflows (a cap of 1): the forces are the reference build's bit for bit.
* Caps between the stacks' needs: some groups overflow after several rounds and far-node
  hand-overs beside groups that do not; the bits are those of the one-wave form, which a
  launch of the same systems beside a large one takes."""
from __future__ import annotations

import numpy as np
import pytest

import galaxy_amd as glx
from galaxy_amd import ic
from galaxy_amd.pool import Pool
from tests import inputs as I

pytestmark = pytest.mark.gpu

BUILDS = {
    "monopole": dict(multipole=0),
    "quadrupole": dict(multipole=2),
    "far": dict(multipole=2, far_theta=0.6, mono_ratio=0.9),
    "kahan_far": dict(multipole=2, far_theta=0.6, precision=glx.PREC_KAHAN),
}


@pytest.mark.parametrize("build", sorted(BUILDS))
@pytest.mark.parametrize("n", [1, 2, 65, 300, 20000])
def test_every_group_overflows(monkeypatch, build, n):
    pos, _, mass = I.cluster(n, n) if n < 1000 else ic.plummer(n, 41)
    prec = BUILDS[build].get("precision", glx.PREC_F32)
    ref = glx.Lbvh(1.0, 0.01, 0.5, precision=prec).accelerations(pos, mass)
    monkeypatch.setenv("GLX_WALK_STACK_CAP", "1")
    s = glx.Lbvh(1.0, 0.01, 0.5, walk=glx.WALK_GROUP, **BUILDS[build])
    assert np.array_equal(s.accelerations(pos, mass), ref)


def states(pool, systems):
    ids = [pool.admit(p, v, m, softening=0.02, theta=0.5, dt=1e-3) for p, v, m in systems]
    for _ in range(2):
        pool.step()
    return [(*pool.snapshot(j), pool.snapshot_accel(j)) for j in ids]


def fallbacks(monkeypatch, cap, system, knobs):
    monkeypatch.setenv("GLX_WALK_STACK_CAP", str(cap))
    s = glx.Lbvh(1.0, 0.02, 0.5, count=True, **knobs)
    s.accelerations(system[0], system[2])
    return s.stats()["fallbacks"]


@pytest.mark.parametrize("cap", [100, 160, 220])
@pytest.mark.parametrize("build", sorted(BUILDS))
def test_some_groups_overflow(monkeypatch, build, cap):
    systems = []
    for n in (200, 1000, 5003):
        pos, vel, mass = I.cluster(n, n, with_vel=True)
        systems.append((pos, vel, mass))
    systems.append(ic.plummer(9001, 5))
    knobs = dict(BUILDS[build], walk=glx.WALK_GROUP)
    groups = fallbacks(monkeypatch, 1, systems[-1], knobs)
    assert 0 < fallbacks(monkeypatch, cap, systems[-1], knobs) < groups
    small = Pool(1 << 30, max_jobs=64, **knobs)
    alone = states(small, systems)
    small.close()
    big = Pool(1 << 30, max_jobs=64, **knobs)
    assert big.admit_ic(ic.spec_plummer(600000, 1), softening=0.02, theta=0.8, dt=1e-3)
    beside = states(big, systems)
    big.close()
    for a, b in zip(alone, beside, strict=True):
        for x, y in zip(a, b, strict=True):
            assert np.array_equal(x, y)
