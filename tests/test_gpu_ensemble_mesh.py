"""The last systems of an ensemble over several workgroups each (run_mesh in
ensemble.cpp): after the first 16 steps of a run, systems of at least 48
sources leave the queue once all of them fit the device.

Compared with the queue alone (SOLARIS_AMD_NO_GRID=1) on RK4 runs, whose steps
do not depend on errors: 48 steps, so that 32 are in the mesh form.  One step's
states agree within 1e-13 (test_gpu_mesh.py); differences grow over 32 steps
of a small fraction of a period by no more than their sum and its growth, ten
times that: 4e-11.  A system that stays in the queue has the same bits.
"""
import os

import numpy as np
import pytest

from solaris_amd import _abi, runtime, scenarios as S

pytestmark = pytest.mark.gpu


def run(scns, integrator, steps, T=1e9, **env):
    env["SOLARIS_AMD_ENSEMBLE_BLOCK"] = "256"
    os.environ.update(env)
    try:
        ens = runtime.Ensemble(scns)
    finally:
        for k in env:
            os.environ.pop(k, None)
    for k, s in enumerate(scns):
        ens.set_system(k, s, _abi.timeline(0.0, s.h_next, T))
    st = ens.run(integrator, 1e-10, max_steps=steps)
    return [ens.get_system(k) for k in range(len(scns))], st, ens.info()


def system(n):
    """A C4 system with n bodies: the first of one with at least n."""
    for k in range(400):
        s = S.make_c4_system(k)
        if s.n >= n:
            break
    s.counts = dict(s.counts)
    s.counts["proto_planet"] = n - 1
    s.counts["total"] = n
    s.y0, s.mass, s.type = s.y0[:n].copy(), s.mass[:n].copy(), s.type[:n].copy()
    s.radius, s.density, s.cd = s.radius[:n].copy(), s.density[:n].copy(), s.cd[:n].copy()
    return s


# sizes of the systems: the least the mesh form takes, and one body
# less (which stays); 7, 15, 23 and 31 bodies per workgroup; more than fit
@pytest.mark.parametrize("sizes", [[47, 48, 257, 5], [257] * 7 + [100], [200] * 14, [257] * 20, [250] * 28,
                                   [120] * 70 + [30] * 10])
def test_rk4_against_the_queue(sizes):
    scns = [system(n) for n in sizes]
    a, sa, ia = run(scns, S.RUNGE_KUTTA4, 48)
    b, sb, ib = run(scns, S.RUNGE_KUTTA4, 48, SOLARIS_AMD_NO_GRID="1")
    assert sa.accepted_steps == sb.accepted_steps == 48 * len(sizes)
    for n, (ya, ta, st, ka), (yb, tb, _, kb) in zip(sizes, a, b):
        assert st == 0 and ka == kb == 48 and ta.time == tb.time and ta.flush_count == tb.flush_count
        assert np.abs(ya - yb).max() <= 4e-11
        assert n >= 48 or np.array_equal(ya, yb)


def test_ends():
    """RKF78 to the end time in the mesh form."""
    scns = [system(n) for n in (50, 90, 150, 257)]
    for T in (20.0, 25.0):
        a, _, _ = run(scns, S.RUNGE_KUTTA_FEHLBERG78, 0, T)
        b, _, _ = run(scns, S.RUNGE_KUTTA_FEHLBERG78, 0, T, SOLARIS_AMD_NO_GRID="1")
        for (ya, ta, st, ka), (yb, tb, _, kb) in zip(a, b):
            assert st == 1 and ta.time == tb.time == T
            assert abs(ka - kb) <= 0.02 * kb + 1 and ka > 16
            assert np.abs(ya[:, :3] - yb[:, :3]).max() <= 1e-8


def test_wait_that_gives_up_stays_in_the_queue():
    """With no wait budget every mesh launch gives up, the systems keep their
    states and the queue's result is what comes out, bit for bit."""
    scns = [system(n) for n in (64, 180, 257)]
    a, _, _ = run(scns, S.RUNGE_KUTTA4, 48, SOLARIS_AMD_GRID_WAIT="0")
    b, _, _ = run(scns, S.RUNGE_KUTTA4, 48, SOLARIS_AMD_NO_GRID="1")
    for (ya, ta, _, ka), (yb, tb, _, kb) in zip(a, b):
        assert ka == kb == 48 and ta.time == tb.time and np.array_equal(ya, yb)
