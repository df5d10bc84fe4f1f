"""The mesh form without a wait budget (SOLARIS_AMD_GRID_WAIT=0): no wait of it
succeeds, however soon the workgroups meet, so each of two calls runs on the
other path from its unchanged start and has that path's bits, as has a caller
loop."""
import numpy as np
import pytest

from solaris_amd import _abi, runtime, scenarios as S

from test_gpu_mesh import DP, RK4, RKF78, make_ctx, other

pytestmark = pytest.mark.gpu


def arrays(ctx):
    return [ctx.get_array(w) for w in (runtime.Y0, runtime.Y, runtime.ACCEL)] + [*ctx.side_outputs()[:3]]


# 5 and 215 workgroups that fall back to one, and 167 to one launch per stage
@pytest.mark.parametrize("n", [34, 1500, 2500])
@pytest.mark.parametrize("integrator", [RKF78, RK4, DP])
def test_same_bits_as_the_other_path(n, integrator):
    scn = S.make_c3(n=n - 1, softening=0.0)
    a, b = make_ctx(scn, SOLARIS_AMD_GRID_WAIT="0"), other(scn)
    print(f"[mesh without a budget, {n} bodies, integrator {integrator}]", flush=True)
    ta, tb = _abi.timeline(0.0, 0.25, 1e12), _abi.timeline(0.0, 0.25, 1e12)
    for _ in range(2):
        assert a.driver(integrator, 1e-10, ta)[0] == 0 and b.driver(integrator, 1e-10, tb)[0] == 0
        assert ta.time == tb.time and ta.hNext == tb.hNext
        for x, y in zip(arrays(a), arrays(b)):
            assert np.array_equal(x, y)
    a, b = make_ctx(scn, SOLARIS_AMD_GRID_WAIT="0"), other(scn)
    (ra, sa), (rb, sb) = (x.integrate(integrator, 1e-10, _abi.timeline(0.0, 0.25, 1e12), max_steps=3) for x in (a, b))
    assert ra == rb == 0 and sa.path == sb.path != _abi.PATH_GRID
    for x, y in zip(arrays(a), arrays(b)):
        assert np.array_equal(x, y)
