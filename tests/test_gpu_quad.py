"""The quad form: whole Driver loops of a system with few sources, four lanes
per body (quad.hip).

Compared with the one-workgroup and per-stage paths (SOLARIS_AMD_NO_GRID=1) at
the sizes where it changes: one to three, four to seven and eight sources (one,
two and three pulls per lane); waves with one body of their own and full ones;
one workgroup and two; the largest system; sink classes of their own source
ranges; events, outputs and the small-number flush; a step that underflows; and
a wait that gives up.  Runs have the same bits as in slices
(SOLARIS_AMD_GRID_BLOCK=64), whose sums the quads follow.

Tolerances as in test_gpu_mesh.py: both sums round to a few 1e-16 per term, so
accelerations agree within the 1e-12 of the force tests, and a state after one
step within h |a| 1e-12 + rounding, far below 1e-13 here (|y| about 1 to 10,
h |a| < 1e-2).
"""
import numpy as np
import pytest

from solaris_amd import _abi, runtime, scenarios as S

from test_gpu_mesh import DP, RK4, RKF78, make_ctx, other, same

pytestmark = pytest.mark.gpu


def system(n, sources, superpl=0, pl=0):
    """The star, `sources` sources (the last `superpl` of them
    super-planetesimals, which pull on the others only), `pl` planetesimals
    and test particles."""
    rng = S.SplitMix64(0x501A00E5)
    groups, counts = [S._star()], dict(central_body=1)
    k0 = sources - superpl
    for key, typ, k, m, lo, hi in (("giant_planet", S.GIANT, min(2, k0), 1e-3, 5.0, 9.0),
                                   ("proto_planet", S.PROTO, max(0, k0 - 2), 1e-6, 1.0, 3.0),
                                   ("super_planetesimal", S.SUPERPL, superpl, 1e-9, 1.0, 3.0),
                                   ("planetesimal", S.PL, pl, 1e-12, 1.0, 4.0),
                                   ("test_particle", S.TP, n - 1 - sources - pl, 0.0, 1.0, 4.0)):
        if k == 0:
            continue
        y = S._orbits(rng, k, 1.0, np.full(k, m), rng.uniform(k, lo, hi), rng.uniform(k, 0.0, 0.1),
                      rng.uniform(k, 0.0, 0.05), massless=(typ == S.TP))
        groups.append(dict(mass=np.full(k, m), type=typ, y0=y, radius=np.full(k, 1e-6), density=np.full(k, 1.0)))
        counts[key] = k
    return S._assemble("few", S._counts(**counts), groups)


def timelines(t=0.0, h=0.25, end=1e12, output=None):
    kw = {} if output is None else dict(output=output)
    return _abi.timeline(t, h, end, **kw), _abi.timeline(t, h, end, **kw)


# (bodies, sources): a wave has 16 - sources of its own, a workgroup four waves
@pytest.mark.parametrize("n,sources", [(3, 2), (3, 1), (4, 2), (18, 2), (59, 2), (60, 2), (70, 1), (17, 3), (56, 4),
                                       (200, 7), (41, 8), (42, 8), (9, 8), (1000, 3), (14339, 2)])
@pytest.mark.parametrize("integrator", [RKF78, RK4, DP])
def test_one_driver_call(n, sources, integrator):
    scn = system(n, sources)
    a, b = make_ctx(scn), other(scn)
    ta, tb = timelines()
    print(f"[quad, {n} bodies, {sources} sources, integrator {integrator}]", flush=True)
    assert a.driver(integrator, 1e-10, ta)[0] == 0 and b.driver(integrator, 1e-10, tb)[0] == 0
    assert ta.hDid == tb.hDid == 0.25
    same(a, b, integrator)
    own = 16 - sources
    _, st = a.integrate(integrator, 1e-10, _abi.timeline(0.0, 0.25, 1e12), max_steps=1)
    assert st.path == _abi.PATH_GRID and st.slices == max(1, -(-(n - 1 - sources) // (4 * own)))


def test_sink_classes_and_source_ranges():
    scn = system(300, 6, superpl=3, pl=40)
    for ranges in (None, (3, 3), (2, 5)):
        a, b = make_ctx(scn), other(scn)
        if ranges:
            a.set_source_ranges(*ranges)
            b.set_source_ranges(*ranges)
        ta, tb = timelines()
        print(f"[quad, sink classes, ranges {ranges}]", flush=True)
        assert a.driver(RKF78, 1e-10, ta)[0] == 0 and b.driver(RKF78, 1e-10, tb)[0] == 0
        same(a, b, RKF78)


@pytest.mark.parametrize("n", [40, 300])
def test_caller_loop_outputs_flush_and_split(n):
    """120 RK4 steps with an output every 10 (the small-number flush comes at
    the 100th), in one call and split at every output."""
    scn = system(n, 2)
    scn.y0[:, 2] = 1e-60
    scn.y0[:, 5] = 0.0
    a, b, c = make_ctx(scn), make_ctx(scn), other(scn)
    ta, tc = timelines(0.0, 0.5, 60.0, 5.0)
    tb, _ = timelines(0.0, 0.5, 60.0, 5.0)
    assert a.integrate(RK4, 0.0, ta)[0] == 0 and c.integrate(RK4, 0.0, tc)[0] == 0
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


@pytest.mark.parametrize("integrator", [RKF78, RK4])
@pytest.mark.parametrize("n", [30, 500])
def test_events(n, integrator):
    scn = system(n, 3)
    q = np.linalg.norm(scn.y0[4:, :3], axis=1)
    settings = (dict(ejection=1.003 * np.linalg.norm(scn.y0[1:, :3], axis=1).max()), dict(hit_centrum=0.999 * q.min()),
                dict(collision_factor=2.0e5))
    for kw in settings:
        a, b = make_ctx(scn), other(scn)
        a.set_events(**kw)
        b.set_events(**kw)
        ta, tb = timelines(0.0, 0.25, 300.0)
        ra, wa, sa = a.integrate_until(integrator, 1e-10, ta, _abi.STOP_EVENT, max_steps=2000)
        rb, wb, sb = b.integrate_until(integrator, 1e-10, tb, _abi.STOP_EVENT, max_steps=2000)
        print(f"[quad, events {kw}] reason {wa} after {sa.accepted_steps} steps", flush=True)
        assert ra == rb == 0 and wa == wb and abs(sa.accepted_steps - sb.accepted_steps) <= 1


def test_underflow():
    scn = system(100, 2)
    a, b = make_ctx(scn), other(scn)
    ta, tb = timelines(1.0e9)
    ra, _ = a.driver(RKF78, 1e-60, ta)
    rb, _ = b.driver(RKF78, 1e-60, tb)
    assert ra == rb != 0 and ta.time == tb.time
    assert np.array_equal(a.get_array(runtime.Y0), b.get_array(runtime.Y0))


def test_wait_that_gives_up_falls_back():
    """With no wait budget the workgroups give up, the call runs on another
    path from its unchanged start, and the result is that path's."""
    scn = system(500, 2)
    a, b = make_ctx(scn, SOLARIS_AMD_GRID_WAIT="0"), other(scn)
    ta, tb = timelines()
    assert a.driver(RKF78, 1e-10, ta)[0] == 0 and b.driver(RKF78, 1e-10, tb)[0] == 0
    assert ta.time == tb.time
    assert np.array_equal(a.get_array(runtime.Y0), b.get_array(runtime.Y0))


def test_many_launches():
    """More RK4 steps than one launch takes, against the same in calls of its
    own, and every workgroup's bodies in a run of one step (without an
    exchange a workgroup may end before another starts)."""
    scn = system(400, 2)
    a, b = make_ctx(scn), make_ctx(scn)
    ta, tb = timelines(0.0, 0.05)
    assert a.integrate(RK4, 0.0, ta, max_steps=21000)[0] == 0
    for k in (9000, 12000):
        assert b.integrate(RK4, 0.0, tb, max_steps=k)[0] == 0
    assert ta.time == tb.time
    assert np.array_equal(a.get_array(runtime.Y0), b.get_array(runtime.Y0))
    scn = system(14339, 2)
    a, b = make_ctx(scn), other(scn)
    ta, tb = timelines(0.0, 0.05)
    for _ in range(20):
        assert a.driver(RK4, 0.0, ta)[0] == 0 and b.driver(RK4, 0.0, tb)[0] == 0
    assert np.abs(a.get_array(runtime.Y0) - b.get_array(runtime.Y0)).max() <= 20 * 1e-13


@pytest.mark.parametrize("n,sources", [(515, 2), (1033, 3), (300, 7), (300, 8)])
@pytest.mark.parametrize("integrator", [RKF78, RK4, DP])
def test_same_bits_as_slices(n, sources, integrator):
    scn = system(n, sources)
    out = []
    for env in ({}, {"SOLARIS_AMD_GRID_BLOCK": "64"}):
        ctx = make_ctx(scn, **env)
        tl = _abi.timeline(0.0, 0.01, 1000.0, output=300.0)
        r, st = ctx.integrate(integrator, 1e-10, tl, max_steps=400)
        assert r == 0 and st.path == _abi.PATH_GRID
        out.append([ctx.get_array(w) for w in (runtime.Y0, runtime.Y, runtime.ACCEL, runtime.ERROR)] +
                   list(ctx.side_outputs()) + [tl.time, tl.hNext, st.attempts])
    print(f"[quad bits, {n} bodies, {sources} sources, integrator {integrator}] {out[0][-1]} attempts", flush=True)
    for x, y in zip(*out):
        assert np.array_equal(x, y)
