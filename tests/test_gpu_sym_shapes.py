"""The symmetric pair sum where its groups and workgroups change: blocks that
end one body into, one body short of and at the end of a group of 256 (and of
a packet of 64), the smallest block, and workgroups of one item and of
several, whose column sums pass from item to item; and the nearest-neighbour
search after the pair sum (up to 8,191 bodies) and beside it.  In mixed
precision also items of four, two and one units, and a change of the precision
of a context, which changes its plan.

FP64 against the one-directional sum (SOLARIS_AMD_NO_SYM=1): both round to a
few 1e-16 of the sum of the terms' magnitudes, within 1e-14 of the total
acceleration as in test_gpu_sym.py.  Mixed precision against FP64 with the
same softening: 1e-7 as there.
"""
import os

import numpy as np
import pytest

from solaris_amd import runtime, scenarios as S

pytestmark = pytest.mark.gpu


def accelerations(scn, precision=0, **env):
    os.environ.update(env)
    try:
        ctx = runtime.Context(scn, precision=precision)
    finally:
        for k in env:
            os.environ.pop(k, None)
    ctx.set_side_outputs(False)
    a = ctx.compute(0.0, scn.y0)[1:, 3:]
    ctx.close()
    return a


def rel(a, b):
    return (np.linalg.norm(a - b, axis=1) / np.linalg.norm(b, axis=1)).max()


# bodies of the block: M - 1
@pytest.mark.parametrize("n", [2048, 2049, 2111, 2112, 2113, 2303, 2304, 2305, 6337, 20481])
@pytest.mark.parametrize("waves", [None, "2", "7"])
def test_fp64_against_one_directional(n, waves):
    scn = S.make_c3(n=n, softening=0.0)
    a = accelerations(scn, **({"SOLARIS_AMD_SYM_WAVES": waves} if waves else {}))
    b = accelerations(scn, SOLARIS_AMD_NO_SYM="1")
    assert rel(a, b) <= 1e-14


@pytest.mark.parametrize("n", [2048, 2049, 2113, 2305, 6337, 7168, 7169, 14336, 14337])
def test_mixed_against_fp64(n):
    scn = S.make_c3(n=n)
    a = accelerations(scn, runtime.MIXED)
    b = accelerations(scn)
    c = accelerations(scn, runtime.MIXED, SOLARIS_AMD_SYM_WAVES="3")
    assert rel(a, b) <= 1e-7 and rel(c, b) <= 1e-7


@pytest.mark.parametrize("n", [8191, 8192])
def test_neighbours_after_and_beside_the_pair_sum(n):
    """Force evaluations one after another, each with its own neighbours; the
    one-directional kernel finds the same ones."""
    scn = S.make_c3(n=n - 1, softening=0.0)
    os.environ["SOLARIS_AMD_NO_SYM"] = "1"
    try:
        plain = runtime.Context(scn)
    finally:
        os.environ.pop("SOLARIS_AMD_NO_SYM")
    ctx = runtime.Context(scn)
    for k in range(3):
        y = scn.y0.copy()
        y[1:, :3] = np.roll(y[1:, :3], k, axis=0)
        a, b = ctx.compute(0.0, y), plain.compute(0.0, y)
        sa, sb = ctx.side_outputs(), plain.side_outputs()
        assert rel(a[1:, 3:], b[1:, 3:]) <= 1e-14
        assert np.array_equal(sa[1], sb[1])
        np.testing.assert_allclose(sa[2], sb[2], rtol=1e-12, atol=0)


def test_change_of_precision():
    scn = S.make_c3(n=6337)
    ctx = runtime.Context(scn, precision=runtime.MIXED)
    ctx.set_side_outputs(False)
    out = []
    for precision in (runtime.MIXED, 0, runtime.MIXED):
        ctx.set_precision(precision, scn.softening)
        out.append(ctx.compute(0.0, scn.y0)[1:, 3:])
    assert np.array_equal(out[0], out[2])
    assert np.array_equal(out[1], accelerations(scn))
    assert rel(out[0], out[1]) <= 1e-7
