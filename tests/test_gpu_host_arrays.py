"""The arrays of a call on their way between the host and the device: through
pinned memory up to 32,768 bodies (the side outputs up to 65,536), copied
above; rows of six doubles in blocks of 256 bodies.

States come back as they went in, to the bit.  A force evaluation and its side
outputs agree with the oracle within the 1e-12 of the other force tests, and
nearest neighbours exactly.
"""
import numpy as np
import pytest

from oracle.cpu_ref import Oracle
from solaris_amd import runtime, scenarios as S

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [3, 255, 256, 257, 32767, 32768, 32769, 65536, 65537])
def test_round_trip_and_compute(n):
    scn = S.make_c1(n_tp=n - 3)
    assert scn.n == n
    ctx = runtime.Context(scn)
    rng = np.random.default_rng(n)
    for which, put in ((runtime.Y0, ctx.set_state), (runtime.ACCEL, ctx.set_accel)):
        v = rng.standard_normal((n, 6))
        put(v)
        assert np.array_equal(ctx.get_array(which), v)
    orc = Oracle(scn)
    for shift in (0.0, 1.0e-3):     # a second call of the same context
        y = scn.y0.copy()
        y[1:, :3] += shift
        a, b = ctx.compute(0.0, y), orc.compute(0.0, y)
        assert np.array_equal(a[:, :3], b[:, :3]) and np.array_equal(a[0], b[0])
        assert (np.linalg.norm(a[1:, 3:] - b[1:, 3:], axis=1) / np.linalg.norm(b[1:, 3:], axis=1)).max() <= 1e-12
        (rm3, nn, dist, mig), (rm3o, nno, disto, migo) = ctx.side_outputs(), orc.side_outputs()
        np.testing.assert_allclose(rm3, rm3o, rtol=1e-12, atol=0)
        np.testing.assert_allclose(dist, disto, rtol=1e-12, atol=0)
        assert np.array_equal(nn, nno) and np.array_equal(mig, migo)
    ctx.close()
