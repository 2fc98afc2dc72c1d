"""k_pairs at the sizes where its mapping has edges: owner groups of one to 64
atoms (batches of owner atoms, classification rounds of fewer entries), passes
whose lane slots straddle groups, atoms with more exclusions than lanes, and
lists short enough to end in the first pass; against the oracle's force at the
tolerances of the other FP64 parity tests (the sums run in another order:
sqrt(pairs) x 1e-16 and the polynomial exponential's 4e-14)."""
import dataclasses

import numpy as np
import pytest

import oracle as O
from conftest import rel, relrms
from test_gpu_parity import E_TOL, F_TOL, _force_gpu, _oracle_list, _stress_close

pytestmark = pytest.mark.gpu


def grouped(sizes, side=12, spacing=2.2, seed=3, many_excluded=False, solute=0.4):
    """side^3 atoms on a jittered lattice, consecutive atoms in groups of the
    given sizes (repeated), one group in three a solute group."""
    from orac_hip import synth
    rng = np.random.default_rng(seed)
    n = side ** 3
    L = side * spacing
    g = (np.arange(side) + 0.5) * spacing - L / 2
    x = np.stack(np.meshgrid(g, g, g, indexing="ij"), -1).reshape(-1, 3) + rng.uniform(-0.2, 0.2, (n, 3))
    first = []
    a = k = 0
    while a < n:
        first.append(a)
        a += sizes[k % len(sizes)]
        k += 1
    first = np.array(first)
    last = np.append(first[1:], n) - 1
    ng = len(first)
    atomg = np.repeat(np.arange(1, ng + 1), last - first + 1).astype(np.int32)
    mass = rng.uniform(1.0, 16.0, n)
    pmass = mass / np.bincount(atomg - 1, weights=mass)[atomg - 1]
    sol = rng.random(ng) < solute
    nt = 5
    tt, e12, e6 = synth._lj_tables(rng.uniform(1.6, 2.4, nt), np.array([0.15, 0.0, 0.1, 0.2, 0.0]))
    cons = np.zeros((2, 0), np.int32)
    if many_excluded:  # atom 1 excludes 100 atoms of other groups, 30 more chain pairs
        far = rng.choice(np.arange(70, n), 100, replace=False)
        cons = np.concatenate([np.stack([np.zeros(100, int), far]),
                               np.stack([np.arange(200, 230), np.arange(201, 231)])], axis=1) + 1
    half = L / 2
    q = rng.normal(0, 0.3, n)
    return synth.System(
        L=L, xp0=x[:, 0] / half, yp0=x[:, 1] / half, zp0=x[:, 2] / half, charge=synth.charge_internal(q - q.mean()),
        mass=mass, nbtype=rng.integers(1, nt + 1, n).astype(np.int32), ntypes=nt, type_table=tt, ecc12=e12, ecc6=e6,
        grppt=np.asfortranarray(np.stack([first + 1, last + 1]).astype(np.int32)), atomg=atomg,
        atomp=atomg.copy(), ss_index=np.where(sol, 1, 2)[atomg - 1].astype(np.int32), pmass=pmass,
        co=np.asfortranarray(np.diag([half] * 3)), oc=np.asfortranarray(np.diag([1 / half] * 3)),
        volume=L ** 3, alpha=0.35, nfft=(24, 24, 24), order=4, rcut=6.0, constraints=cons.astype(np.int32))


CASES = {
    "singles": dict(sizes=[1]),
    "waters": dict(sizes=[3]),
    "four": dict(sizes=[4]),
    "mixed": dict(sizes=[1, 3, 2, 5, 1, 4]),
    "seven_one": dict(sizes=[7, 1, 1]),
    "largest": dict(sizes=[64, 1, 3, 17]),
    "exclusions": dict(sizes=[1, 3], many_excluded=True),
    "few": dict(sizes=[3, 1], side=5, spacing=4.0),
    # around a mean of eight atoms a group, where owners take eight atoms a list walk
    "eight": dict(sizes=[8]),
    "nine": dict(sizes=[9]),
    "full": dict(sizes=[64]),
    "tails": dict(sizes=[17, 8, 64, 3, 10, 1]),
    "large_excluded": dict(sizes=[16, 7], many_excluded=True),
}


@pytest.mark.parametrize("shell", ["single", "outer", "plain"])
@pytest.mark.parametrize("name", list(CASES))
def test_force_forms(gpu_ctx, name, shell):
    s = grouped(**CASES[name])
    nnlpp, fa, _ = _oracle_list(s)
    kw = dict(rinn=0.0, rout=s.rcut, rtolinn=0.0, rtolout=s.rtol, rneigh=0.0)
    if shell == "outer":
        kw.update(rinn=3.5, rtolinn=0.4, lskip_ewald=True)
    elif shell == "plain":
        kw.update(lskip_ewald=True, ewald=False)
    g = _force_gpu(gpu_ctx, s, nnlpp, fa, **kw)
    o = O.force(s, nnlpp, fa=fa, **kw)
    assert relrms(g["f"], o["f"]) < F_TOL
    for k in ("uconf_slt", "uconf_slv", "uconf_ss", "ucoul_slt", "ucoul_slv", "ucoul_ss"):
        scale = max(abs(o[k]), 1e-3 * abs(o["uconf_ss"]) + 1e-3 * abs(o["ucoul_ss"]))  # sums of both signs cancel
        assert abs(g[k] - o[k]) <= E_TOL * max(scale, 1e-300), k
    assert _stress_close(g["stress"], o["stress"])


@pytest.mark.parametrize("name", ["mixed", "largest", "exclusions", "nine", "tails", "large_excluded"])
def test_mixed_precision_forms(gpu_ctx, name):
    """The FP32 pair form on the same groups: forces within the mixed-precision bar of FP64."""
    from orac_hip.api import ResidentSystem
    s = grouped(**CASES[name])
    f = []
    for precision in (0, 1):
        rs = ResidentSystem(gpu_ctx, s, precision=precision)
        rs.eval()
        f.append(rs.results())
        rs.close()
    assert relrms(f[1]["f"], f[0]["f"]) < 5e-6
    assert rel(f[1]["uconf_ss"], f[0]["uconf_ss"]) < 1e-5


@pytest.mark.parametrize("precision", [0, 1])
def test_large_and_small_groups_in_one_batch(gpu_ctx, precision):
    """Systems whose owners take three and eight atoms a list walk, and an
    alchemical one of each, in one launch: each gets what it gets alone."""
    from orac_hip import synth
    from orac_hip.api import Batch, ResidentSystem
    systems = [grouped(sizes=z, seed=k) for k, z in enumerate(([3], [9], [17, 8, 64, 3, 10, 1], [1, 2]))]
    for alchemical in ((), (0, 2)):
        rss = [ResidentSystem(gpu_ctx, s, precision=precision) for s in systems]
        alone = []
        for k, (s, rs) in enumerate(zip(systems, rss)):
            if k in alchemical:
                rs.set_alchemy(synth.alchemy_for(s, np.arange(40)), synth.lambda_state(0.4, lrm0=0.5))
            rs.eval(rebuild_list=True)
            alone.append(rs.results())
        b = Batch(gpu_ctx, rss)
        for persistent in (0, 1):
            b.set_tuning(persistent=persistent)
            b.eval(rebuild_list=True)
            for r, a in zip(b.results(), alone):
                assert np.array_equal(r["f"], a["f"]) and r["uconf_ss"] == a["uconf_ss"]
                assert np.array_equal(r["stress"], a["stress"])
        b.close()
        for rs in rss:
            rs.close()


@pytest.mark.parametrize("name", ["waters", "nine", "tails"])
def test_alchemical_forms_at_full_coupling(gpu_ctx, name):
    """At lambda = 0 the soft core is the plain pair: the alchemical form of any
    group size gives the plain form's forces."""
    from orac_hip import synth
    from orac_hip.api import ResidentSystem
    s = grouped(**CASES[name])
    rs = ResidentSystem(gpu_ctx, s)
    rs.eval()
    plain = rs.results()["f"]
    # (mixed types by sigma and epsilon of each atom, as the system's own tables are)
    rs.set_alchemy(synth.alchemy_for(s, np.arange(0, s.natoms, 3)), synth.lambda_state(0.0))
    rs.eval()
    f = rs.results()["f"]
    rs.close()
    assert relrms(f, plain) < F_TOL


@pytest.mark.parametrize("name", ["mixed", "nine", "tails"])
def test_rem_forms(gpu_ctx, name):
    from test_gpu_rem import _check, _force_rem_gpu
    s = grouped(**CASES[name])
    nnlpp, fa, _ = _oracle_list(s)
    rem = (np.random.default_rng(4).random(s.natoms) < 0.2).astype(np.int32)
    kw = dict(rinn=3.5, rout=s.rcut, rtolinn=0.4, rtolout=s.rtol, rneigh=0.0)
    g = _force_rem_gpu(gpu_ctx, s, nnlpp, fa, rem, 2, 0.55, **kw)
    _check(g, O.force_rem(s, nnlpp, rem, rem_kind=2, rem_f3=0.55, fa=fa, **kw))


def test_owner_atoms_order(gpu_ctx):
    """Groups in another order than their atoms: owners and neighbours are found by their records."""
    s = grouped(sizes=[3, 1, 2])
    p = np.random.default_rng(1).permutation(s.ngrp)
    inv = np.argsort(p)
    s2 = dataclasses.replace(s, grppt=np.asfortranarray(s.grppt[:, p]), atomg=(inv[s.atomg - 1] + 1).astype(np.int32))
    nnlpp, fa, _ = _oracle_list(s2)
    kw = dict(rinn=0.0, rout=s.rcut, rtolinn=0.0, rtolout=s.rtol, rneigh=0.0)
    g = _force_gpu(gpu_ctx, s2, nnlpp, fa, **kw)
    o = O.force(s2, nnlpp, fa=fa, **kw)
    assert relrms(g["f"], o["f"]) < F_TOL
    assert _stress_close(g["stress"], o["stress"])


@pytest.mark.parametrize("ngrp", [1, 2, 64, 65, 130, 216])
def test_half_list_transpose(gpu_ctx, water216, ngrp):
    """Every pair of the first ngrp groups listed (group i lists all j > i, in
    descending order): reverse lists of 0 to ngrp - 1 entries, around the 64
    lanes of the transpose's sort; forces against the oracle on the same list."""
    s = water216
    nnlpp = np.concatenate([np.concatenate([[max(0, ngrp - i)], np.arange(ngrp, i, -1)]) if i <= ngrp else [0]
                            for i in range(1, s.ngrp + 1)]).astype(np.int32)
    fa = O.ForceArgs(s)
    kw = dict(rinn=0.0, rout=s.rcut, rtolinn=0.0, rtolout=s.rtol, rneigh=0.0)
    g = _force_gpu(gpu_ctx, s, nnlpp, fa, **kw)
    o = O.force(s, nnlpp, fa=fa, **kw)
    assert np.abs(g["f"] - o["f"]).max() <= F_TOL * max(np.abs(o["f"]).max(), 1e-300)
    assert _stress_close(g["stress"], o["stress"])


@pytest.mark.parametrize("precision", [0, 1])
def test_coincident_atoms_spoil_their_own_forces_only(gpu_ctx, precision):
    """Two atoms of different groups at one point have no finite force; the other
    atoms of their groups do (within the switching range alone a group pair's
    energy enters the forces of all its atoms), so that a relaxation can move them."""
    from orac_hip.api import ResidentSystem
    s = grouped(sizes=[3])
    # the third atoms of the first group and of its neighbour along y
    x = [np.array(v) for v in (s.xp0, s.yp0, s.zp0)]
    for v in x:
        v[14] = v[2]
    t = s.nbtype.copy()
    t[[2, 14]] = 1  # (a type with LJ: r^-12 overflows FP32)
    s = dataclasses.replace(s, xp0=x[0], yp0=x[1], zp0=x[2], nbtype=t)
    rs = ResidentSystem(gpu_ctx, s, precision=precision)
    rs.eval()
    f = rs.results()["f"]
    rs.close()
    bad = np.flatnonzero(~np.isfinite(f).all(axis=0)).tolist()
    # (FP64 leaves a distance of its rounding between them, and a force of 1e200)
    assert bad == [2, 14] if precision == 1 else set(bad) <= {2, 14}
