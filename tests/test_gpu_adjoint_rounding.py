"""The rounding of the adjoint's forward pass (adjoint_few.hip): bodies that
start at rest end one very short RK4 step with v = h a, all four stages at the
same positions, so the error of |v| is the rounding of |r|^-3 and of a few
products around it.  The exact step is the same one in 80 bits.

Three accelerations: the star's, a planet's pull on a body near it, and the
indirect term of a planet on a far one.

Bound: the root mean square over the bodies of the relative error along the
velocity, in units of 2^-53.  Emulated in double precision (every product and
sum rounded as here, the reciprocal square root good to 2^-27) it is 1.34, 1.39
and 1.22 for 1 / (r^2 sqrt(r^2)), 1.16, 1.26 and 1.15 for a corrected cube and
1.55, 1.72 and 1.68 for the cube of a rounded reciprocal square root, so 1.4 holds
the first two and not the third.
"""
import dataclasses

import numpy as np
import pytest

from solaris_amd import runtime, scenarios as S

pytestmark = pytest.mark.gpu

H = 2.0**-27          # displacements of less than half a unit in the last place


def exact(gm0, gmp, y, h):
    """One RK4 step of (planet, sinks) at rest in 80 bits; the sinks' velocities."""
    L = np.longdouble
    x0, v0 = y[:, :3].astype(L), y[:, 3:].astype(L)

    def acc(x):
        rm3 = 1 / ((x * x).sum(1) ** L(1.5))
        mu = np.full(len(x), L(gm0))
        mu[0] = L(np.float64(gm0) + np.float64(gmp))
        a = -(mu * rm3)[:, None] * x
        d = x[0] - x[1:]
        a[1:] += L(gmp) * (d / ((d * d).sum(1) ** L(1.5))[:, None] - x[0] * rm3[0])
        return a

    h = L(h)
    k1 = acc(x0)
    k2 = acc(x0 + h / 2 * v0)
    k3 = acc(x0 + h / 2 * (v0 + h / 2 * k1))
    k4 = acc(x0 + h * (v0 + h / 2 * k2))
    return (v0 + h * (k1 + 2 * k2 + 2 * k3 + k4) / 6)[1:]


def relative(d, want):
    return (d * want).sum(1) / (want * want).sum(1) * 2.0**53


def errors(star, planet, xp, xs):
    """Relative errors of the sinks' velocities along them, in units of 2^-53."""
    scn = S.make_c5(n_tp=len(xs), n_pl=1)
    mass = np.zeros(scn.n)
    mass[0], mass[1] = star, planet
    y0 = np.zeros((scn.n, 6))
    y0[1, :3], y0[2:, :3] = xp, xs
    scn = dataclasses.replace(scn, mass=mass, y0=y0)
    ctx = runtime.Context(scn)
    ctx.set_state(y0)
    y = ctx.adjoint_forward(0.0, 0.0, 1, 1, h_seq=np.array([H]))
    ctx.close()
    want = exact(S.GAUSS2 * star, S.GAUSS2 * planet, y0[1:], H)
    d = (y[2:, 3:].astype(np.longdouble) - want).astype(float)
    return relative(d, want.astype(float))


def directions(rng, n):
    v = rng.normal(size=(n, 3))
    return v / np.linalg.norm(v, axis=1)[:, None]


@pytest.mark.parametrize("term", ["star", "pair", "indirect"])
def test_rounding(term):
    rng = np.random.RandomState(11)
    if term == "star":
        xs = directions(rng, 2000) * np.exp(rng.uniform(np.log(0.5), np.log(30.0), 2000))[:, None]
        e = errors(1.0, 1e-22, [200.0, 10.0, 1.0], xs)
    elif term == "pair":
        xp = np.array([0.8, -0.5, 0.1])
        xs = xp + directions(rng, 2000) * np.exp(rng.uniform(np.log(0.2), np.log(0.5), 2000))[:, None]
        e = errors(1e-22, 1.0, xp, xs)
    else:
        e = np.concatenate([errors(1e-22, 1.0, directions(rng, 1)[0] * np.exp(rng.uniform(np.log(0.5), np.log(5.0))),
                                   directions(rng, 1) * 1e9) for _ in range(300)])
    rms = np.sqrt((e * e).mean())
    print(f"[adjoint forward, {term}: {rms:.2f} rms, {abs(e).max():.2f} largest, in units of 2^-53]", flush=True)
    assert rms <= 1.4
