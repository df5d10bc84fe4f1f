"""Members of an ensemble beside others and alone: with the mesh form off
(SOLARIS_AMD_NO_GRID=1) and a fixed launch shape of one body per thread the
results have the same bits, as the header says; with the mesh form on, a member
that it takes agrees with itself in the queue within what test_gpu_ensemble_mesh.py
allows, and the same ensemble run again has the same bits."""
import numpy as np
import pytest

from solaris_amd import scenarios as S

from test_gpu_ensemble_mesh import run, system

pytestmark = pytest.mark.gpu

SIZES = [5, 30, 48, 60, 96, 97, 150, 257]


@pytest.mark.parametrize("integrator", [S.RUNGE_KUTTA_FEHLBERG78, S.RUNGE_KUTTA4, S.DORMAND_PRINCE])
def test_alone_and_in_company(integrator):
    scns = [system(n) for n in SIZES]
    together, _, _ = run(scns, integrator, 40, SOLARIS_AMD_NO_GRID="1")
    for scn, (y, tl, status, steps) in zip(scns, together):
        ((ya, ta, sa, ka),), _, _ = run([scn], integrator, 40, SOLARIS_AMD_NO_GRID="1")
        assert (sa, ka) == (status, steps) and ta.time == tl.time and ta.hNext == tl.hNext
        assert np.array_equal(ya, y)


def test_again():
    scns = [system(n) for n in SIZES]
    a, _, _ = run(scns, S.RUNGE_KUTTA4, 48)
    b, _, _ = run(scns, S.RUNGE_KUTTA4, 48)
    c, _, _ = run(scns, S.RUNGE_KUTTA4, 48, SOLARIS_AMD_NO_GRID="1")
    for (ya, *_), (yb, *_), (yc, *_) in zip(a, b, c):
        assert np.array_equal(ya, yb)
        assert np.abs(ya - yc).max() <= 4e-11
