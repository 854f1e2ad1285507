"""Downloads when pinned lanes run short: more threads than the process has lanes (each waits
its turn), and none to be had at all (GLX_DOWNLOAD_LANES=0 caps them), where snapshots come
through plain copies instead. Every download returns what was uploaded."""
from __future__ import annotations

import threading

import numpy as np
import pytest

import galaxy_amd as glx
from galaxy_amd.pool import Pool

pytestmark = pytest.mark.gpu


def state(n, seed):
    r = np.random.default_rng(seed)
    vel = r.standard_normal((n, 3)).astype(np.float32).astype(np.float64)  # as they are held
    return r.standard_normal((n, 3)), vel, r.uniform(0.5, 1.5, n)


def check(got, want):
    for g, w in zip(got, want, strict=True):
        assert np.array_equal(g, w)


def resident(r):
    s = r.snapshot()
    return s.pos, s.vel, s.mass


def test_more_threads_than_lanes():
    """12 handles at once, up to four lanes each, of at most 8."""
    count = 12
    gate = threading.Barrier(count)
    errs, done = [], []

    def one(k):
        try:
            want = state(470_001 if k % 2 else 150_001, k)
            r = glx.GpuResidentLeapfrog(1.0, 0.05, 0.5)
            r.upload(*want)
            for _ in range(3):
                gate.wait(timeout=60)
                check(resident(r), want)
            r.close()
            done.append(k)
        except BaseException as e:  # reported in the main thread
            gate.abort()
            errs.append(e)

    ts = [threading.Thread(target=one, args=(k,), daemon=True) for k in range(count)]
    for t in ts:
        t.start()
    for t in ts:
        t.join(timeout=100)
    assert not errs, errs
    assert not any(t.is_alive() for t in ts)
    assert sorted(done) == list(range(count))


@pytest.mark.parametrize("lanes", ["0", "1", "2"])
@pytest.mark.parametrize("n", [1, 43_691, 87_382, 470_001])
def test_few_or_no_lanes(monkeypatch, lanes, n):
    monkeypatch.setenv("GLX_DOWNLOAD_LANES", lanes)
    want = state(n, n)
    r = glx.GpuResidentLeapfrog(1.0, 0.05, 0.5)
    r.upload(*want)
    check(resident(r), want)
    r.step(1e-3)  # a later kernel launch reports no error left behind
    acc = r.snapshot_accel()
    r.close()
    p = Pool(1 << 30)
    job = p.admit(*want, softening=0.05, theta=0.5, dt=1e-3)
    check((*p.snapshot(job), p.snapshot_mass(job)), want)
    p.close()
    monkeypatch.delenv("GLX_DOWNLOAD_LANES")
    r = glx.GpuResidentLeapfrog(1.0, 0.05, 0.5)
    r.upload(*want)
    r.step(1e-3)
    assert np.array_equal(r.snapshot_accel(), acc)
    r.close()


def test_handles_one_after_the_other():
    """The lanes come with the first 4 MiB of a handle's life and go with the last handle;
    small snapshots before that are plain copies."""
    for n in (1, 2_000, 470_001, 2_000, 150_001):
        want = state(n, n)
        r = glx.GpuResidentLeapfrog(1.0, 0.05, 0.5)
        r.upload(*want)
        for _ in range(1 + min(200, (6 << 20) // (60 * n))):
            check(resident(r), want)
        r.close()
