"""The mesh form: whole Driver loops of a self-gravitating system shared out
over workgroups that exchange positions at every stage (mesh.hip).

Compared with the one-workgroup and per-stage paths
(SOLARIS_AMD_NO_GRID=1), which sum the same pair terms in another order, at
the sizes where the shares change: 7 bodies per workgroup up to 1,793, then
15 to 3,841 and 23 to 5,889; the smallest system it takes; sink
classes of their own source ranges; events, outputs and the small-number
flush; a step that underflows; and a wait that gives up.

Tolerances: both sums round to a few 1e-16 per term, so accelerations agree
within the 1e-12 of the force tests, and a state after one step within
h |a| 1e-12 + rounding, far below 1e-13 here (|y| about 1, h |a| < 1e-2).
"""
import os

import numpy as np
import pytest

from solaris_amd import _abi, runtime, scenarios as S

pytestmark = pytest.mark.gpu

RKF78, RK4, DP = S.RUNGE_KUTTA_FEHLBERG78, S.RUNGE_KUTTA4, S.DORMAND_PRINCE


def make_ctx(scn, **env):
    os.environ.update(env)
    try:
        ctx = runtime.Context(scn)
    finally:
        for k in env:
            os.environ.pop(k, None)
    ctx.set_state(scn.y0)
    return ctx


def other(scn):
    return make_ctx(scn, SOLARIS_AMD_NO_GRID="1")


def same(a, b, integrator):
    """State, previous state, derivative and side outputs after one call."""
    for which in (runtime.Y0, runtime.Y):
        assert np.abs(a.get_array(which) - b.get_array(which)).max() <= 1e-13
    fa, fb = a.get_array(runtime.ACCEL), b.get_array(runtime.ACCEL)
    norm = np.linalg.norm(fb[1:, 3:], axis=1)
    assert (np.linalg.norm(fa[1:, 3:] - fb[1:, 3:], axis=1) / norm).max() <= 1e-12
    if integrator == RKF78:
        np.testing.assert_allclose(a.get_array(runtime.YSCALE), b.get_array(runtime.YSCALE), rtol=1e-12)
    sa, sb = a.side_outputs(), b.side_outputs()
    np.testing.assert_allclose(sa[0][1:], sb[0][1:], rtol=1e-12)
    assert np.array_equal(sa[1][1:], sb[1][1:])
    np.testing.assert_allclose(sa[2][1:], sb[2][1:], rtol=0, atol=1e-13)


@pytest.mark.parametrize("n", [34, 66, 514, 1793, 1794, 3842, 5889])
@pytest.mark.parametrize("integrator", [RKF78, RK4, DP])
def test_one_driver_call(n, integrator):
    scn = S.make_c3(n=n - 1, softening=0.0)
    a, b = make_ctx(scn), other(scn)
    ta, tb = _abi.timeline(0.0, 0.25, 1e12), _abi.timeline(0.0, 0.25, 1e12)
    print(f"[mesh, {n} bodies, integrator {integrator}]", flush=True)
    assert a.driver(integrator, 1e-10, ta)[0] == 0 and b.driver(integrator, 1e-10, tb)[0] == 0
    assert ta.hDid == tb.hDid == 0.25
    same(a, b, integrator)
    _, st = a.integrate(integrator, 1e-10, _abi.timeline(0.0, 0.25, 1e12), max_steps=1)
    assert st.path == _abi.PATH_GRID


def sink_classes(n_proto):
    rng = S.SplitMix64(0x501A00E3)
    groups, counts = [S._star()], dict(central_body=1)
    for key, typ, k, m in (("giant_planet", S.GIANT, 3, 1e-4), ("proto_planet", S.PROTO, n_proto, 1e-9),
                           ("super_planetesimal", S.SUPERPL, 37, 1e-10), ("planetesimal", S.PL, 61, 1e-12),
                           ("test_particle", S.TP, 50, 0.0)):
        y = S._orbits(rng, k, 1.0, np.full(k, m), rng.uniform(k, 1.0, 8.0), rng.uniform(k, 0.0, 0.1),
                      rng.uniform(k, 0.0, 0.05), massless=(typ == S.TP))
        groups.append(dict(mass=np.full(k, m), type=typ, y0=y, radius=np.full(k, 1e-6), density=np.full(k, 1.0)))
        counts[key] = k
    return S._assemble("classes", S._counts(**counts), groups)


@pytest.mark.parametrize("n_proto", [90, 2000])
def test_sink_classes_and_source_ranges(n_proto):
    scn = sink_classes(n_proto)
    for ranges in (None, (scn.n, scn.n), (scn.n_massive(), 40)):
        a, b = make_ctx(scn), other(scn)
        if ranges:
            a.set_source_ranges(*ranges)
            b.set_source_ranges(*ranges)
        ta, tb = _abi.timeline(0.0, 0.25, 1e12), _abi.timeline(0.0, 0.25, 1e12)
        print(f"[mesh, sink classes, {scn.n} bodies, ranges {ranges}]", flush=True)
        assert a.driver(RKF78, 1e-10, ta)[0] == 0 and b.driver(RKF78, 1e-10, tb)[0] == 0
        same(a, b, RKF78)


def test_softening():
    scn = S.make_c3(n=300, softening=1e-2)
    a, b = make_ctx(scn), other(scn)
    ta, tb = _abi.timeline(0.0, 0.25, 1e12), _abi.timeline(0.0, 0.25, 1e12)
    assert a.driver(RKF78, 1e-10, ta)[0] == 0 and b.driver(RKF78, 1e-10, tb)[0] == 0
    same(a, b, RKF78)


def test_caller_loop_outputs_flush_and_split():
    """120 RK4 steps with an output every 10 (the small-number flush comes at
    the 100th), in one call and split at every output."""
    scn = S.make_c3(n=40, softening=0.0)
    scn.y0[:, 2] = 1e-60
    scn.y0[:, 5] = 0.0
    a, b, c = make_ctx(scn), make_ctx(scn), other(scn)
    ta, tc = (_abi.timeline(0.0, 0.5, 60.0, output=5.0) for _ in range(2))
    assert a.integrate(RK4, 0.0, ta)[0] == 0 and c.integrate(RK4, 0.0, tc)[0] == 0
    tb = _abi.timeline(0.0, 0.5, 60.0, output=5.0)
    stops = 0
    while True:
        r, why, _ = b.integrate_until(RK4, 0.0, tb, _abi.STOP_OUTPUT)
        assert r == 0
        stops += 1
        if why & _abi.STOP_END:
            break
    assert stops == 12 and ta.time == tb.time == tc.time == 60.0
    ya, yb, yc = (x.get_array(runtime.Y0) for x in (a, b, c))
    assert np.array_equal(ya, yb)
    assert np.abs(ya - yc).max() <= 1e-12
    assert np.all(np.abs(yc[1:, 2]) < 1e-50) and np.all(np.abs(ya[1:, 2]) < 1e-50)


def test_events():
    scn = S.make_c3(n=200, softening=0.0)
    scn.radius[1:] = 1e-3
    a, b = make_ctx(scn), other(scn)
    for x in (a, b):
        x.set_events(ejection=6.0, hit_centrum=0.1, collision_factor=8.0)
    ta, tb = _abi.timeline(0.0, 0.25, 300.0), _abi.timeline(0.0, 0.25, 300.0)
    ra, wa, sa = a.integrate_until(RKF78, 1e-10, ta, _abi.STOP_EVENT)
    rb, wb, sb = b.integrate_until(RKF78, 1e-10, tb, _abi.STOP_EVENT)
    assert ra == rb == 0 and wa == wb and sa.accepted_steps == sb.accepted_steps
    assert wa & _abi.STOP_EVENT


def test_underflow():
    scn = S.make_c3(n=100, softening=0.0)
    a, b = make_ctx(scn), other(scn)
    ta, tb = _abi.timeline(1.0e9, 0.25, 1e12), _abi.timeline(1.0e9, 0.25, 1e12)
    ra, _ = a.driver(RKF78, 1e-60, ta)
    rb, _ = b.driver(RKF78, 1e-60, tb)
    assert ra == rb != 0 and ta.time == tb.time
    assert np.array_equal(a.get_array(runtime.Y0), b.get_array(runtime.Y0))


def test_wait_that_gives_up_falls_back():
    """With no wait budget the workgroups give up, the call runs on another
    path from its unchanged start, and the result is that path's."""
    scn = S.make_c3(n=1500, softening=0.0)
    a, b = make_ctx(scn, SOLARIS_AMD_GRID_WAIT="0"), other(scn)
    ta, tb = _abi.timeline(0.0, 0.25, 1e12), _abi.timeline(0.0, 0.25, 1e12)
    assert a.driver(RK4, 0.0, ta)[0] == 0 and b.driver(RK4, 0.0, tb)[0] == 0
    assert ta.time == tb.time
    assert np.abs(a.get_array(runtime.Y0) - b.get_array(runtime.Y0)).max() <= 1e-13
