"""The RK4 adjoint of systems with few sources (adjoint_few.hip) where its
shape changes: the numbers of sources at the edges of its eight lanes and of
its workgroup, the last one it takes (32) and the first it leaves (33); a
system of sources alone; sinks of different source ranges; steps at the edges
of its chunks of 64; stage states kept and recomputed.

Against the launch-by-launch products (SOLARIS_AMD_VJP_WIDE=1), which form
the same terms in another order: states and gradients within 1e-12 of the
largest entry, the bound the products are held to against each other, over
steps short enough that no close encounter amplifies the rounding.
"""
import numpy as np
import pytest

from solaris_amd import runtime, scenarios as S

pytestmark = pytest.mark.gpu


def gradient(scn, hs, k, ranges=None):
    ctx = runtime.Context(scn)
    if ranges:
        ctx.set_source_ranges(*ranges)
    ctx.set_state(scn.y0)
    y = ctx.adjoint_forward(0.0, 0.0, len(hs), k, h_seq=hs)
    g = np.zeros_like(y)
    g[1:] = np.random.RandomState(3).normal(size=(scn.n - 1, 6))
    out = (y,) + tuple(ctx.adjoint_backward(g))
    ctx.close()
    return out


def compare(monkeypatch, scn, steps, ranges=None):
    hs = 0.02 + 0.01 * (np.arange(steps) % 3)
    monkeypatch.setenv("SOLARIS_AMD_VJP_WIDE", "1")
    want = gradient(scn, hs, 50, ranges)
    monkeypatch.setenv("SOLARIS_AMD_VJP_WIDE", "0")
    got = gradient(scn, hs, 50, ranges)
    monkeypatch.setenv("SOLARIS_AMD_ADJOINT_RECORD_MB", "0")
    again = gradient(scn, hs, 37, ranges)
    for a, b, c in zip(got, want, again):
        assert np.abs(a - b).max() <= 1e-12 * np.abs(b).max()
        assert np.array_equal(a, c)


@pytest.mark.parametrize("sources", [1, 2, 7, 8, 9, 16, 17, 32, 33])
def test_sources(sources, monkeypatch):
    print(f"[adjoint, {sources} sources]", flush=True)
    compare(monkeypatch, S.make_c5(n_tp=203, n_pl=sources, seed=0x501A0105), 10)


@pytest.mark.parametrize("steps", [1, 63, 64, 65, 129])
def test_steps(steps, monkeypatch):
    print(f"[adjoint, {steps} steps]", flush=True)
    compare(monkeypatch, S.make_c5(n_tp=70, n_pl=5, seed=0x501A0105), steps)


def test_sources_alone(monkeypatch):
    scn = S.make_c3(n=9, softening=0.0)
    compare(monkeypatch, scn, 20)


def test_sink_classes(monkeypatch):
    """Planets that see the super-planetesimals, planetesimals that do not,
    and ranges by hand that leave some sources unseen by one class."""
    rng = S.SplitMix64(0x501A00C7)
    groups, counts = [S._star()], dict(central_body=1)
    for key, typ, k, m in (("giant_planet", S.GIANT, 2, 1e-4), ("proto_planet", S.PROTO, 5, 1e-6),
                           ("super_planetesimal", S.SUPERPL, 4, 1e-8), ("planetesimal", S.PL, 90, 1e-12)):
        y = S._orbits(rng, k, 1.0, np.full(k, m), rng.uniform(k, 1.0, 8.0), rng.uniform(k, 0.0, 0.1),
                      rng.uniform(k, 0.0, 0.05))
        groups.append(dict(mass=np.full(k, m), type=typ, y0=y, radius=np.full(k, 1e-6), density=np.full(k, 1.0)))
        counts[key] = k
    scn = S._assemble("classes", S._counts(**counts), groups)
    for ranges in (None, (5, 20), (20, 3)):
        compare(monkeypatch, scn, 12, ranges)
