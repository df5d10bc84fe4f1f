"""A profiled context keeps the launches that are timed: small Dormand-Prince
systems with gas, which neither a workgroup nor the slices take, run in quads
otherwise (quad.hip)."""
import numpy as np
import pytest

from solaris_amd import _abi, runtime, scenarios as S

from test_gpu_mesh import DP, RKF78, make_ctx, same

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n_pl,planets", [(20, 1), (120, 4)])
def test_launches_are_timed(n_pl, planets):
    scn = S.make_c2(n_pl=n_pl, n_proto=planets)
    a, b = make_ctx(scn), make_ctx(scn)
    b.profile(True)
    for ctx in (a, b):
        tl = _abi.timeline(0.0, 0.25, 1e12)
        for _ in range(3):
            assert ctx.driver(DP, 1e-9, tl)[0] == 0
            tl.hNext = 0.25
    prof = b.profile(False)
    print(f"[profiled, {scn.n} bodies: {prof.epilogue_launches} epilogues, {prof.epilogue_ms:.3f} ms]", flush=True)
    # the first evaluation and eight stages of three steps
    assert prof.epilogue_launches == 27
    assert prof.pair_launches + prof.pair_nn_launches == 27
    assert prof.epilogue_ms > 0.0
    same(a, b, DP)
    # forms that time nothing stay
    b.profile(True)
    tl = _abi.timeline(0.0, 0.25, 1e12)
    _, st = b.integrate(RKF78, 1e-9, tl, max_steps=1)
    assert st.path == _abi.PATH_GRID and b.profile(False).epilogue_launches == 0
    _, st = b.integrate(DP, 1e-9, tl, max_steps=1)
    assert st.path == _abi.PATH_GRID
