"""The fast level of a step (launch_md_advance) where its mapping has edges:
units without terms, sets of atoms connected by terms around the slots of a
workgroup (one, two a thread, too many for one), small sets sharing
workgroups, atoms of many terms, terms that reach rigid units; against
oracle.md_steps at the tolerance of the other dynamics tests, on atoms without
nonbonded forces, so that these terms and constraints are all that acts."""
import ctypes as C
import dataclasses

import numpy as np
import pytest

import oracle as O
from test_gpu_spread_forms import _random

pytestmark = pytest.mark.gpu


def _chain(first, n):
    return [(first + k, first + k + 1) for k in range(n - 1)] + [(first + k, first + k + 2) for k in range(n - 2)]


# atoms, rigid units' first atoms, terms (0-based)
CASES = {
    "free": (70, [0, 5, 8, 66], []),
    "pairs": (1500, [0, 1490], [(k, k + 1) for k in range(4, 1480, 2)]),
    "chains": (2000, [1990], _chain(0, 700) + _chain(700, 400) + _chain(1100, 64) + _chain(1164, 1)),
    "chain1024": (1030, [1025], _chain(0, 1024)),
    "chain1025": (1030, [1026], _chain(0, 1025)),
    "chain2048": (2053, [2049], _chain(0, 2048)),
    "chain2049": (2060, [2050, 2054], _chain(0, 2049)),
    "hub": (200, [190], [(100, k) for k in range(100)] + _chain(101, 60)),
    "on_rigid": (300, [0, 10, 20, 30], _chain(40, 100) + [(12, 13), (31, 200), (200, 201), (201, 202)]),
}


def _make(ctx, name, seed=5):
    from orac_hip.api import ResidentSystem, _check, _f, _i, _p, lib
    n, first, terms = CASES[name]
    rng = np.random.default_rng(seed)
    s = _random(n=n, nfft=(20, 20, 20), order=4, L=40.0)
    x = rng.uniform(-18.0, 18.0, (3, n))
    lens = np.tile([1.1, 1.2, 1.7], (len(first), 1))
    cosa = (1.1 ** 2 + 1.2 ** 2 - 1.7 ** 2) / (2 * 1.1 * 1.2)
    for a in first:
        e = np.linalg.qr(rng.normal(size=(3, 3)))[0]
        x[:, a + 1] = x[:, a] + 1.1 * e[:, 0]
        x[:, a + 2] = x[:, a] + 1.2 * (cosa * e[:, 0] + np.sqrt(1 - cosa ** 2) * e[:, 1])
    mass = rng.uniform(1.0, 16.0, n)
    xp = np.asarray(s.oc) @ x
    s = dataclasses.replace(s, xp0=xp[0], yp0=xp[1], zp0=xp[2], mass=mass, charge=0.0 * s.charge, rcut=5.0,
                            ecc12=0.0 * s.ecc12, ecc6=0.0 * s.ecc6)
    pairs = np.array(terms, np.int32).reshape(-1, 2).T + 1
    d = x[:, pairs[0] - 1] - x[:, pairs[1] - 1]
    k = rng.uniform(0.002, 0.02, pairs.shape[1])
    r0 = np.sqrt((d * d).sum(0)) * rng.uniform(0.97, 1.03, pairs.shape[1])
    f1 = np.array(first, np.int32) + 1
    rs = ResidentSystem(ctx, s, precision=0)
    keep = (_i(f1), _f(lens.ravel()), _i(pairs.T.ravel() if pairs.size else np.zeros(2)), _f(np.append(k, 0.0)),
            _f(np.append(r0, 1.0)))
    a, b, c, e, f = keep
    _check(lib().orac_hip_md_setup(ctx._h, rs.id, C.c_int32(len(first)), _p(a), _p(b), C.c_int32(pairs.shape[1]), _p(c),
                                   _p(e), _p(f)))
    v = rng.normal(0, 0.01, (3, n))
    rs.keep = keep
    return rs, s, x, v, pairs, k, r0, (f1, lens)


def _start(rs, x, v):
    from orac_hip.api import _check, _f, _p, lib
    a = [_f(q) for q in (*x, *v)]
    _check(lib().orac_hip_md_set_state(rs.ctx._h, rs.id, *[_p(q) for q in a]))
    return _state(rs)


def _state(rs):
    from orac_hip.api import _check, _p, lib
    arr = [np.zeros(rs.natoms) for _ in range(6)]
    _check(lib().orac_hip_md_get_state(rs.ctx._h, rs.id, *[_p(q) for q in arr]))
    return np.stack(arr[:3]), np.stack(arr[3:])


@pytest.mark.parametrize("name", list(CASES))
def test_fast_level(gpu_ctx, name):
    from orac_hip import md
    from orac_hip.api import Batch
    rs, s, x, v, pairs, k, r0, (f1, lens) = _make(gpu_ctx, name)
    b = Batch(gpu_ctx, [rs])
    runs = []
    for graph, parts in ((False, [4]), (True, [4]), (True, [1, 3]), (False, [3, 1])):
        x0, v0 = _start(rs, x, v)
        for p in parts:
            md.run_batch(b, p, dt=2.0, ninner=3, list_every=2, graph=graph)
        runs.append(_state(rs))
    for xr, vr in runs[1:]:
        assert np.array_equal(xr, runs[0][0]) and np.array_equal(vr, runs[0][1])
    b.close()
    rs.close()
    cons = O.constraint_tables(f1, lens, s.mass)
    zero = lambda q: np.zeros_like(q)
    xo, vo, fails = O.md_steps(x0, v0, s.mass, 4, 2.0, 3, zero, lambda q: O.harmonic_forces(q, pairs, k, r0), cons)
    assert fails == 0 and np.abs(xo - x0).max() > 1e-2
    assert np.abs(runs[0][0] - xo).max() <= 1e-9
    assert np.abs(runs[0][1] - vo).max() <= 1e-9 * np.abs(vo).max()


def test_fast_level_batch(gpu_ctx):
    """All of these in one batch: each system's trajectory alone, bit for bit."""
    from orac_hip import md
    from orac_hip.api import Batch
    made = [_make(gpu_ctx, name) for name in CASES]
    alone = []
    for m in made:
        _start(m[0], m[2], m[3])
        b = Batch(gpu_ctx, [m[0]])
        md.run_batch(b, 2, dt=2.0, ninner=3, list_every=2)
        b.close()
        alone.append(_state(m[0]))
    for m in made:
        _start(m[0], m[2], m[3])
    b = Batch(gpu_ctx, [m[0] for m in made])
    md.run_batch(b, 2, dt=2.0, ninner=3, list_every=2)
    b.close()
    for m, (xa, va) in zip(made, alone):
        xb, vb = _state(m[0])
        assert np.array_equal(xa, xb) and np.array_equal(va, vb)
        m[0].close()


@pytest.mark.parametrize("n", [1, 87381, 87382])
def test_state_read_back(gpu_ctx, n):
    """Positions and velocities come back as set, through the staging memory
    up to its size (6 x 87,381 doubles) and past it; records of closed systems
    start clean for the next ones."""
    from orac_hip.api import ResidentSystem, _check, _f, _i, _p, lib
    s = _random(n=n, nfft=(40, 40, 40), order=4, L=110.0)
    for k in range(2):
        rs = ResidentSystem(gpu_ctx, s, precision=0)
        r = rs.results()
        assert r["eer"] == 0.0  # (the list is counted already)
        z = (_i(np.zeros(2)), _f(np.zeros(2)))
        _check(lib().orac_hip_md_setup(gpu_ctx._h, rs.id, C.c_int32(0), _p(z[0]), _p(z[1]), C.c_int32(0), _p(z[0]),
                                       _p(z[1]), _p(z[1])))
        rng = np.random.default_rng(k)
        x, v = rng.uniform(-50, 50, (3, n)), rng.normal(size=(3, n))
        xs, vs = _start(rs, x, v)
        assert np.array_equal(x, xs) and np.array_equal(v, vs)
        rs.eval(rebuild_list=True)
        assert n == 1 or rs.results()["f"].any()
        rs.close()
