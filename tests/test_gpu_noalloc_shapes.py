"""sol_compute_gravity_noalloc at the sizes where its launch changes: a sink
per thread for few sources, else 7, 15, 23 or 31 sinks per workgroup with the
sources in LDS tiles of 1,024; sink classes of different source ranges in one
system; and y and dydt the same array.

Against sol_compute, whose pair sums round in another order: accelerations
within 1e-12 relative per body, the bound of the force tests.
"""
import ctypes as C

import numpy as np
import pytest
import torch

from solaris_amd import _abi, runtime, scenarios as S

pytestmark = pytest.mark.gpu


def call(scn, in_place=False):
    lib = runtime.library()
    nb = _abi.nbodies(scn.counts)
    y = torch.from_numpy(scn.y0.copy()).cuda()
    m = torch.from_numpy(np.ascontiguousarray(scn.mass)).cuda()
    out = y if in_place else torch.full_like(y, float("nan"))
    err = C.create_string_buffer(256)
    stream = torch.cuda.current_stream().cuda_stream
    r = lib.sol_compute_gravity_noalloc(C.byref(nb), y.data_ptr(), m.data_ptr(), out.data_ptr(), stream, err, 256)
    assert r == 0, err.value
    return out.cpu().numpy()


def check(scn, in_place=False):
    ctx = runtime.Context(scn)
    want = ctx.compute(0.0, scn.y0)
    ctx.close()
    got = call(scn, in_place)
    assert np.array_equal(got[:, :3], want[:, :3]) and np.all(got[0] == 0.0)
    norm = np.linalg.norm(want[1:, 3:], axis=1)
    assert (np.linalg.norm(got[1:, 3:] - want[1:, 3:], axis=1) / norm).max() <= 1e-12


@pytest.mark.parametrize("n", [2, 9, 10, 64, 66, 1025, 1026, 1793, 1794, 3841, 4097, 5889, 5890, 12001])
def test_mutual_bodies(n):
    print(f"[noalloc, {n} mutually attracting bodies]", flush=True)
    check(S.make_c3(n=n - 1, softening=0.0))


@pytest.mark.parametrize("planets,particles", [(2, 1), (7, 300), (40, 300), (40, 12000), (63, 70), (64, 20000)])
def test_few_sources(planets, particles):
    print(f"[noalloc, {planets} planets, {particles} particles]", flush=True)
    check(S.make_c5(n_tp=particles, n_pl=planets))


@pytest.mark.parametrize("n_proto,n_super,n_pl", [(30, 20, 500), (300, 1, 100), (1500, 600, 900)])
def test_sink_classes_in_place(n_proto, n_super, n_pl):
    rng = S.SplitMix64(0x501A00D1)
    groups, counts = [S._star()], dict(central_body=1)
    for key, typ, k, m in (("giant_planet", S.GIANT, 2, 1e-4), ("proto_planet", S.PROTO, n_proto, 1e-9),
                           ("super_planetesimal", S.SUPERPL, n_super, 1e-10), ("planetesimal", S.PL, n_pl, 1e-12)):
        y = S._orbits(rng, k, 1.0, np.full(k, m), rng.uniform(k, 1.0, 8.0), rng.uniform(k, 0.0, 0.1),
                      rng.uniform(k, 0.0, 0.05))
        groups.append(dict(mass=np.full(k, m), type=typ, y0=y, radius=np.full(k, 1e-6), density=np.full(k, 1.0)))
        counts[key] = k
    scn = S._assemble("classes", S._counts(**counts), groups)
    print(f"[noalloc, sink classes, {scn.n} bodies]", flush=True)
    check(scn)
    check(scn, in_place=True)
