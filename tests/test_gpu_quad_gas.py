"""The quad form with gas (quad.hip): drag and migration, four lanes per body,
in the slices of the grid form.

Compared with one launch per stage (SOLARIS_AMD_NO_GRID=1 and
SOLARIS_AMD_NO_RESIDENT=1) for one Driver call: slices of 64 and 128 places, one
to eight planets, the last slice with one body; the three drag regimes and the
density inside the inner edge; exponents that are whole quarters and others; a
nebula that decays; Type I and Type II migration and one that stops.

Tolerances as in test_gpu_quad.py: the drag is rounded differently by some
1e-12 of itself (most of it cancellation) and at most 1e-2 of the pull, so
accelerations agree within 1e-12, or 1e-13 where the drag is as weak as usual;
states after one step within 1e-13.
"""
import copy

import numpy as np
import pytest

from solaris_amd import _abi, runtime, scenarios as S

from test_gpu_mesh import DP, RK4, RKF78, make_ctx, same

pytestmark = pytest.mark.gpu


def pair(scn):
    return make_ctx(scn), make_ctx(scn, SOLARIS_AMD_NO_GRID="1", SOLARIS_AMD_NO_RESIDENT="1")


def check(scn, integrator, calls=1, h=0.25):
    a, b = pair(scn)
    ta, tb = _abi.timeline(3.0, h, 1e12), _abi.timeline(3.0, h, 1e12)
    for _ in range(calls):
        assert a.driver(integrator, 1e-9, ta)[0] == 0 and b.driver(integrator, 1e-9, tb)[0] == 0
        ta.hNext = tb.hNext = h
        assert ta.hDid == tb.hDid == h
    same(a, b, integrator)
    assert np.array_equal(a.side_outputs()[3], b.side_outputs()[3])
    # the caches: the drag of the last stage and the migration of the first
    for x in (a, b):
        x.set_evaluate(0, 0, 0)
    fa, fb = a.compute(3.0, scn.y0), b.compute(3.0, scn.y0)
    assert (np.linalg.norm(fa[1:, 3:] - fb[1:, 3:], axis=1) / np.linalg.norm(fb[1:, 3:], axis=1)).max() <= 1e-12
    _, st = a.integrate(integrator, 1e-9, _abi.timeline(3.0, h, 1e12), max_steps=1)
    assert st.path == _abi.PATH_GRID
    return st


# (planetesimals, planets): slices of 64 - 1 - planets, above 160 of them 128 - 1 - planets
@pytest.mark.parametrize("n_pl,planets", [(125, 4), (177, 4), (178, 4), (61 * 2, 2), (300, 1), (300, 3), (500, 7),
                                          (500, 8), (9600, 4)])
@pytest.mark.parametrize("integrator", [RKF78, RK4, DP])
def test_one_driver_call(n_pl, planets, integrator):
    scn = S.make_c2(n_pl=n_pl, n_proto=planets)
    print(f"[quad gas, {n_pl} planetesimals, {planets} planets, integrator {integrator}]", flush=True)
    st = check(scn, integrator)
    places = 64 if -(-n_pl // (63 - planets)) <= 160 else 128
    assert st.slices == -(-n_pl // (places - 1 - planets))


def changed(**kw):
    scn = S.make_c2(n_pl=300, n_proto=4)
    scn.gas = copy.deepcopy(scn.gas)
    scn.gas.update(kw)
    return scn


@pytest.mark.parametrize("gas", [dict(mean_free_path=(1e-3, 2.75)), dict(mean_free_path=(4.6e-12, 2.75)),
                                 dict(density=(0.002, -2.6)), dict(eta=(0.0019, 0.55), scale_height=(0.05, 1.25)),
                                 dict(scale_height=(0.05, 4.25)), dict(inner_edge=2.0),
                                 dict(type=2, time_scale=10.0), dict(type=1, t0=1.0, t1=9.0)])
@pytest.mark.parametrize("integrator", [RKF78, DP])
def test_nebula(gas, integrator):
    scn = changed(**gas)
    if "mean_free_path" in gas:
        scn.radius = scn.radius.copy()
        scn.radius[5:] *= np.logspace(-3, 3, scn.n - 5)
    print(f"[quad gas, {gas}]", flush=True)
    check(scn, integrator)


def test_migration_that_stops_and_type_ii():
    scn = S.make_c2(n_pl=300, n_proto=4)
    scn.mig_stop_at = scn.mig_stop_at.copy()
    r = np.linalg.norm(scn.y0[1:5, :3], axis=1)
    scn.mig_stop_at[1] = 1.01 * r[0]        # stops at once
    check(scn, RK4, calls=3)
    giants = S.make_c2(n_pl=300, n_proto=4)
    giants.counts = dict(giants.counts)
    giants.counts["giant_planet"], giants.counts["proto_planet"] = 2, 2
    giants.type = giants.type.copy()
    giants.type[1:3] = S.GIANT
    giants.mig_type = giants.mig_type.copy()
    giants.mig_type[1:3] = S.MIG_II
    check(giants, RKF78)
    check(giants, RK4, calls=2)


def test_split_run_is_the_same():
    """RK4 steps in one call and one by one: the caches and types carry over."""
    scn = S.make_c2(n_pl=400, n_proto=3)
    a, b = make_ctx(scn), make_ctx(scn)
    ta, tb = _abi.timeline(0.0, 0.25, 1e12), _abi.timeline(0.0, 0.25, 1e12)
    assert a.integrate(RK4, 0.0, ta, max_steps=12)[0] == 0
    for _ in range(4):
        assert b.integrate(RK4, 0.0, tb, max_steps=3)[0] == 0
    assert ta.time == tb.time
    for which in (runtime.Y0, runtime.Y, runtime.ACCEL):
        assert np.array_equal(a.get_array(which), b.get_array(which))


@pytest.mark.parametrize("n_pl,planets", [(128, 1), (178, 4), (500, 8), (9600, 4)])
@pytest.mark.parametrize("integrator", [RKF78, RK4, DP])
def test_same_bits_as_slices_in_a_thin_nebula(n_pl, planets, integrator):
    """A drag too weak to change any sum leaves the pulls, with the slices' bits."""
    scn = S.make_c2(n_pl=n_pl, n_proto=planets)
    scn.gas = copy.deepcopy(scn.gas)
    scn.gas.update(density=(1e-60, -2.75))
    out = []
    for env in ({}, dict(SOLARIS_AMD_GRID_BLOCK="128")):
        ctx = make_ctx(scn, **env)
        tl = _abi.timeline(0.0, 0.25, 1e12)
        r, st = ctx.integrate(integrator, 1e-10, tl, max_steps=12)
        assert r == 0 and st.path == _abi.PATH_GRID
        out.append([ctx.get_array(w) for w in (runtime.Y0, runtime.Y, runtime.ACCEL)] + [*ctx.side_outputs()[:3], tl.hNext])
    for x, y in zip(*out):
        assert np.array_equal(x, y)
