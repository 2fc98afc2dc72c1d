"""Performance cases of the force library: what its users have it do.

Three ways of use are covered, each through its public entry points:

* resident systems and batches (``orac_hip.api.ResidentSystem``, ``Batch``):
  a full force evaluation with a list rebuild, replayed from the batch's
  graph, with the energies read after it and the forces left on the device,
  for one system, for Hamiltonian replicas and for lambda windows;
* dynamics (``orac_hip.md``): a chunk of outer r-RESPA steps of one system or
  of a served batch, with one or two nonbonded shells, and the state read at
  its end;
* the drop-in calls an ORAC build makes with host arrays (``lc_list`` +
  ``force``, ``fft_pme``).

``exact`` restates the evaluation in 64 bits with torch and numpy (group-pair
search by brute force, numpy FFTs).  Trajectories have no ``exact``: their
end state hangs on the stopping rule of the constraint iteration.
"""
import functools
import math
import os
import sys

import numpy as np
import torch

_ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
if os.path.join(_ROOT, "orac-porting_amd") not in sys.path:
    sys.path.insert(0, os.path.join(_ROOT, "orac-porting_amd"))

import ctypes as C  # noqa: E402

from orac_hip import api, md, serve, synth  # noqa: E402

# ---------------------------------------------------------------- cases


def listed():
    return [
        # one small box, double precision: launch latency, what a water test or a tiny request sees
        dict(name="eval_water648_fp64", kind="eval", system="water", size=6, rcut=8.5, order=5, precision=0,
             replicas=1),
        # the benchmark's solvated solute (24,460 atoms, one LJ type per solute atom), plain double precision
        dict(name="eval_solvated24k_fp64", kind="eval", system="solvated", size=1660, rcut=10.0, order=5, precision=0,
             replicas=1),
        # the same in mixed precision
        dict(name="eval_solvated24k_mixed", kind="eval", system="solvated", size=1660, rcut=10.0, order=5,
             precision=1, replicas=1),
        # a large serving request: a 20,000-atom solute in water (103k atoms), grid 108^3
        dict(name="eval_request103k_mixed", kind="eval", system="request", size=20000, rcut=9.5, order=5, precision=1,
             replicas=1),
        # Hamiltonian replicas of the solvated solute, one launch per stage for all
        dict(name="eval_hrem16_mixed", kind="eval", system="solvated", size=1660, rcut=10.0, order=5, precision=1,
             replicas=16),
        # 16 lambda windows of a ligand in water with their dU/dlambda steps
        dict(name="windows16_mixed", kind="windows", size=48, replicas=16, rcut=9.0, order=5, precision=1),
        # dynamics of the small water box: every launch and every gap counts
        dict(name="md_water648_fp64", kind="md", system="water", size=6, rcut=8.5, order=5, precision=0, replicas=1,
             steps=20, shells=False),
        # dynamics of one solvated request, double precision, lists every 5 steps
        dict(name="md_request16k_fp64", kind="md", system="request", size=1660, rcut=9.5, order=5, precision=0,
             replicas=1, steps=10, shells=False),
        # the same with the nonbonded forces split in two shells
        dict(name="md_shells16k_fp64", kind="md", system="request", size=1660, rcut=9.5, order=5, precision=0,
             replicas=1, steps=5, shells=True),
        # a served batch of eight requests of 9,458 atoms in mixed precision
        dict(name="md_served8_mixed", kind="md", system="request", size=500, rcut=9.5, order=5, precision=1,
             replicas=8, steps=10, shells=False),
        # ORAC's own calls with host arrays: reciprocal sum ...
        dict(name="call_fft_pme16k", kind="fft_pme", system="request", size=1660, rcut=9.5, order=5, precision=0,
             replicas=1),
        # ... and linked-cell list + direct sum
        dict(name="call_direct16k", kind="direct", system="request", size=1660, rcut=9.5, order=5, precision=0,
             replicas=1),
    ]


def draw(rng):
    """One more case: water boxes of 216 to 17,576 molecules, requests of 60 to
    20,000 solute atoms, the solvated solute; spline orders 4 to 6, cut-offs
    8.5 to 10.5 A, both precisions, one to 16 systems."""
    kind = rng.choice(["eval", "eval", "eval", "md", "md", "windows", "fft_pme", "direct"])
    rcut = round(rng.uniform(8.5, 10.5), 2)
    order = rng.choice([4, 5, 5, 6])
    if kind == "windows":
        return dict(kind=kind, size=rng.randint(20, 60), replicas=rng.randint(2, 16),
                    rcut=round(rng.uniform(8.5, 9.5), 2), order=order, precision=rng.randint(0, 1))
    precision = 0 if kind in ("fft_pme", "direct") else rng.randint(0, 1)
    system = rng.choice(["water", "request"])
    atoms = math.exp(rng.uniform(math.log(700), math.log(50000 if precision == 0 else 100000)))
    if kind == "md":
        atoms = min(atoms, 16000)
    if system == "water":
        size = max(6, min(26, int(round((atoms / 3.0) ** (1.0 / 3.0)))))
        rcut = min(rcut, 0.5 * size * 3.1067 - 0.7)
        atoms = 3 * size ** 3
    else:
        size = max(60, int(math.exp(rng.uniform(math.log(60), math.log(max(61.0, atoms / 5.0))))))
        atoms = min(atoms, 30 * size + 7000)
    c = dict(kind=kind, system=system, size=size, rcut=round(rcut, 2), order=order, precision=precision, replicas=1)
    if kind in ("eval", "md") and atoms < 25000:
        c["replicas"] = rng.choice([1, 1, rng.randint(2, 12 if kind == "eval" else 6)])
    if kind == "md":
        c["shells"] = rng.random() < 0.3
        c["steps"] = max(2, min(10, int((40000 if c["shells"] else 80000) / (atoms * c["replicas"]))))
    return c


# ---------------------------------------------------------------- systems

_ALPHA = 0.35
_DT = 1.0        # fs, outer step of the dynamics (2 x _DT with two shells)
_NINNER = 4
_LIST_EVERY = 5
_SHELL = (5.0, 0.5)


def _system(case, seed, k):
    """System k of a case, from the seed alone."""
    sd = 1000003 * (int(seed) % 65521) + 7919 * k + 11
    if case["system"] == "water":
        n = case["size"]
        L = 3.1067 * n
        K = serve.fft_size(max(L, 20.0))
        return synth.water_box(seed=sd, L=L, nside=n, alpha=0.40, nfft=(K, K, K), order=case["order"],
                               rcut=case["rcut"])
    if case["system"] == "solvated":
        # one solute, its own water placement per seed and replica; replicas scale the solute's charges and wells
        s = synth.hrem_scales(case["replicas"])[k]
        return synth.solvated_solute(seed=sd, solute_seed=1001, n_solute=case["size"], order=case["order"],
                                     rcut=case["rcut"], charge_scale=float(s), eps_scale=float(s))
    return serve.serving_request(sd, case["size"], rcut=case["rcut"], alpha=_ALPHA, order=case["order"])


def _windows(case, seed):
    sd = 1000003 * (int(seed) % 65521) + 29
    return synth.alchemy_windows(n_windows=case["replicas"], seed=sd, n_ligand=case["size"], order=case["order"],
                                 rcut=case["rcut"])


def _corr_pairs(s):
    """The solute's flexible 1-2 and 1-3 pairs (per-step reciprocal corrections)."""
    if s.bonds is None:
        return np.zeros((2, 0), np.int32)
    return np.concatenate([s.bonds, s.bends], axis=1)


class _Dev:
    """Device memory of a resident system for torch (keeps the system's context alive)."""

    def __init__(self, ptr, n, keep):
        self.keep = keep
        self.__cuda_array_interface__ = dict(shape=(n,), typestr="<f8", data=(ptr, False), version=2)


def _forces(rs):
    p = [C.c_void_p() for _ in range(3)]
    api._check(api.lib().orac_hip_system_device_ptrs(rs.ctx._h, rs.id, None, None, None, *[C.byref(v) for v in p]))
    return [torch.as_tensor(_Dev(v.value, rs.natoms, rs.ctx), device="cuda") for v in p]


def _energies(rs):
    """Energies, stress and list size of the last evaluation (the forces stay on the device)."""
    e = np.zeros(21)
    api._check(api.lib().orac_hip_system_results(rs.ctx._h, rs.id, None, None, None, e.ctypes.data_as(C.c_void_p)))
    return dict(energies=np.concatenate([e[:9], e[19:]]), stress=e[9:18].reshape(3, 3, order="F"), entries=int(e[18]))


def prepare(case, seed):
    kind = case["kind"]
    ctx = api.Context(0)
    if kind in ("fft_pme", "direct"):
        return _prepare_call(case, seed, ctx)
    if kind == "windows":
        s, al, states = _windows(case, seed)
        rss = []
        for lam in states:
            rs = api.ResidentSystem(ctx, s, precision=case["precision"], corr_pairs=_corr_pairs(s))
            rs.set_alchemy(al, lam)
            rss.append(rs)
        return dict(case=case, ctx=ctx, rss=rss, batch=api.Batch(ctx, rss), f=[_forces(r) for r in rss])
    systems = [_system(case, seed, k) for k in range(case["replicas"])]
    if kind == "eval":
        rss = [api.ResidentSystem(ctx, s, precision=case["precision"], corr_pairs=_corr_pairs(s)) for s in systems]
        return dict(case=case, ctx=ctx, rss=rss, batch=api.Batch(ctx, rss), f=[_forces(r) for r in rss])
    # dynamics: positions relaxed in double precision, velocities at 300 K from the seed
    rss, dyns = [], []
    for k, s in enumerate(systems):
        rs = api.ResidentSystem(ctx, s, precision=0, corr_pairs=_corr_pairs(s))
        d = md.Dynamics(rs, s)
        b = api.Batch(ctx, [rs])
        md.relax_batch(b, 80, dmax=0.05)
        x = d.state()[0]
        b.close()
        if case["precision"] or case["shells"]:
            if case["precision"]:
                rs.close()
                rs = api.ResidentSystem(ctx, s, precision=1, corr_pairs=_corr_pairs(s))
            if case["shells"]:
                rs.set_shells(*_SHELL)
            d = md.Dynamics(rs, s)
        d.set_positions(x)
        d.maxwell_boltzmann(300.0, int(seed) % 65521 + 101 * k)
        rss.append(rs)
        dyns.append(d)
    batch = api.Batch(ctx, rss)
    return dict(case=case, ctx=ctx, rss=rss, dyns=dyns, batch=batch)


def _prepare_call(case, seed, ctx):
    s = _system(case, seed, 0)
    st = dict(case=case, ctx=ctx, s=s, xpcm=s.molecule_coms(), xpg=s.group_centres(), mapnl=s.mapnl())
    if case["kind"] == "fft_pme":
        ctx.fft_pme_init(s.natoms, *s.nfft, s.order)
    else:
        rc = s.rcut + s.rtol + s.rnei
        nc = max(3, int(s.L // 3.5))
        try:
            st["sten"] = ctx.lc_index(4096, nc, nc, nc, rc, s.co)
        except api.OracHipError:  # a box below three list cut-offs takes one cell
            nc = 1
            st["sten"] = ctx.lc_index(4096, 1, 1, 1, rc, s.co)
        st["nc"] = nc
        st["nnlpp"] = np.zeros(s.ngrp * 240 + 1024, np.int32)
    return st


def run(state):
    case, kind = state["case"], state["case"]["kind"]
    if kind == "fft_pme":
        s, n = state["s"], state["s"].natoms
        f = [np.zeros(n) for _ in range(3)]
        stress = np.zeros((3, 3), order="F")
        eer = state["ctx"].fft_pme(n, s.xp0, s.yp0, s.zp0, *state["xpcm"], s.charge, s.co, s.oc, s.volume, s.alpha,
                                   s.order, *s.nfft, *f, stress, s.atomp, s.grppt, True, 1.0e9)
        return dict(f=f, eer=eer, stress=stress)
    if kind == "direct":
        s, n, nc = state["s"], state["s"].natoms, state["nc"]
        nind, ii, jj, kk = state["sten"]
        xpg = state["xpg"]
        f = [np.zeros(n) for _ in range(3)]
        stress = np.zeros((3, 3), order="F")
        state["ctx"].lc_list(nc, nc, nc, nind, ii, jj, kk, s.rcut + s.rtol + s.rnei, s.co, *xpg, s.ngrp,
                             state["nnlpp"])
        e = state["ctx"].force(s.ss_index, s.xp0, s.yp0, s.zp0, *xpg, s.charge, s.nbtype, s.type_table, s.ntypes, n,
                               s.atomg, *state["xpcm"], None, s.atomp, s.co, s.ecc12, s.ecc6, s.alpha,
                               state["mapnl"], s.ngrp, s.grppt, *f, stress, state["nnlpp"], np.zeros(8, np.int32),
                               0.0, 0.0, s.rcut, 0.0, s.rtol, s.pmass, 1, s.mass, synth.MASSINFTY, False, True)
        return dict(f=f, energies=np.array([e[k] for k in api.ENERGY_FIELDS[1:7]]), stress=stress,
                    list=state["nnlpp"])
    if kind == "md":
        kw = dict(dt=_DT, ninner=_NINNER, list_every=_LIST_EVERY)
        if case["shells"]:
            kw.update(dt=2.0 * _DT, nmid=2, ninner=2)
        md.run_batch(state["batch"], case["steps"], **kw)
        out = [d.state() for d in state["dyns"]]
        return dict(x=[o[0] for o in out], v=[o[1] for o in out])
    state["batch"].eval(rebuild_list=True, graph=True)
    out = dict(f=state["f"], system=[_energies(r) for r in state["rss"]])
    if case["replicas"] > 8:  # many systems: their records side by side
        e = out["system"]
        out["system"] = dict(energies=np.stack([v["energies"] for v in e]), stress=np.stack([v["stress"] for v in e]),
                             entries=np.array([v["entries"] for v in e]))
    if kind == "windows":
        a = [r.alchemy_results() for r in state["rss"]]
        out["dwrk"] = np.array([[v[k] for k in _DW] for v in a])
    return out


_DW = ("dwrk", "direct", "recip", "corr", "self", "eer0")

# ---------------------------------------------------------------- work and tolerance


@functools.lru_cache(maxsize=64)
def _size(system, size, rcut, order, replicas):
    s = _system(dict(system=system, size=size, rcut=rcut, order=order, replicas=replicas), 1, 0)
    return s.natoms, s.volume, s.nfft[0], s.rcut + s.rtol


def work(case):
    if case["kind"] == "windows":
        n, vol, k, rc = 3 * 2117 + case["size"], 40.0 ** 3, 48, case["rcut"] + 0.3
    else:
        n, vol, k, rc = _size(case["system"], case["size"], case["rcut"], case["order"], 1)
    g, p3 = k ** 3, case["order"] ** 3
    pairs = 0.5 * n * (4.0 / 3.0 * math.pi * rc ** 3) * n / vol
    direct = 89.0 * pairs                                            # flops per pair within the cut-off
    recip = 8.0 * p3 * n + 2 * 2.5 * g * math.log2(g) + 10.0 * g     # spread + gather, two real transforms, convolution
    # coordinates, charge, type in; forces out; the neighbour relation and the grids live inside the call
    b = (24 + 8 + 4 + 24) * n
    kind = case["kind"]
    if kind == "fft_pme":
        return dict(bytes=float(b), flops=recip)
    if kind == "direct":
        return dict(bytes=float(b), flops=direct)
    reps = case["replicas"]
    if kind == "windows":
        return dict(bytes=float(b * reps), flops=reps * (direct + 1.5 * recip))
    if kind == "md":
        reps *= case["steps"]
        b += 2 * 24 * n
    return dict(bytes=float(b * reps), flops=reps * (direct + recip))


def tolerance(case):
    """FP64: the same sums in another order and with another exponential
    (against 64 bits the forces are off by 4e-15 to 2e-13, 3e-10 in windows
    whose soft-core terms nearly cancel; other summation orders move a
    trajectory by 3e-14).  Mixed precision: FP32 pair terms, splines and
    transforms, summed in FP64 (off by 2e-7 to 1e-6)."""
    if case["precision"]:
        return dict(rel=1e-5) if case["kind"] == "md" else dict(rel=4e-6)
    if case["kind"] in ("md", "windows"):
        return dict(rel=2e-11) if case["kind"] == "md" else dict(rel=1e-9)
    return dict(rel=2e-12)


# ---------------------------------------------------------------- the evaluation in 64 bits

_A = (0.2548296, -0.28449674, 1.4214137, -1.453152, 1.0614054)  # Abramowitz & Stegun 7.1.26
_P = 0.3275911
_PI32 = float(np.float32(math.pi))


def _erfc(x):
    t = 1.0 / (1.0 + _P * x)
    e = torch.exp(-x * x)
    return ((((_A[4] * t + _A[3]) * t + _A[2]) * t + _A[1]) * t + _A[0]) * t * e, e


def _t(a, dev):
    return torch.as_tensor(np.ascontiguousarray(a), device=dev)


def _direct(s, dev, al=None, lam=None, want_list=0.0):
    """Group-switched Ewald erfc + LJ (or soft-core) sum over all group pairs."""
    n, ng = s.natoms, s.ngrp
    co = _t(np.array(s.co), dev)
    x = torch.stack([_t(c, dev) for c in (s.xp0, s.yp0, s.zp0)], 1)
    q, typ, ss = _t(s.charge, dev), _t(s.nbtype.astype(np.int64) - 1, dev), _t(s.ss_index.astype(np.int64), dev)
    mass, mol = _t(s.mass, dev), _t(s.atomp.astype(np.int64) - 1, dev)
    ag = _t(s.atomg.astype(np.int64) - 1, dev)
    g0 = _t(s.grppt[0].astype(np.int64) - 1, dev)
    gn = _t((s.grppt[1] - s.grppt[0] + 1).astype(np.int64), dev)
    zero3 = lambda m: torch.zeros(m, 3, dtype=torch.float64, device=dev)  # noqa: E731
    mg = torch.zeros(ng, dtype=torch.float64, device=dev).index_add_(0, ag, mass)
    w = mass / mg[ag]
    xg = zero3(ng).index_add_(0, ag, w[:, None] * x)
    nmol = int(s.atomp.max())
    mm = torch.zeros(nmol, dtype=torch.float64, device=dev).index_add_(0, mol, mass)
    xm = zero3(nmol).index_add_(0, mol, mass[:, None] * x) / mm[:, None]
    ex = s.exclusion_pairs().astype(np.int64)
    keys = _t(np.unique(np.minimum(ex[0], ex[1]) * (n + 1) + np.maximum(ex[0], ex[1])), dev)
    lij = _t(s.type_table.astype(np.int64) - 1, dev)
    e12, e6 = _t(s.ecc12, dev), _t(s.ecc6, dev)
    if al is not None:
        rmin, eps, ssa = _t(al.rmin, dev), _t(al.epsm, dev), _t(al.ss_alchemy.astype(np.int64), dev)
        ladd, lrm, ladd0, lrm0, laddq, lrmq, laddq0, lrmq0 = [abs(float(v)) for v in lam]
    rout, tol = s.rcut, s.rtol
    rout0 = rout + tol
    f = zero3(n)
    en = torch.zeros(6, dtype=torch.float64, device=dev)
    st = torch.zeros(3, 3, dtype=torch.float64, device=dev)
    dw = torch.zeros((), dtype=torch.float64, device=dev)
    entries = 0
    kmax = int(gn.max())
    rows = max(1, int(3e7 // ng))
    for r0 in range(0, ng, rows):
        r1 = min(ng, r0 + rows)
        d = xg[r0:r1, None, :] - xg[None, :, :]
        sh = 2.0 * torch.round(0.5 * d)
        d = (d - sh) @ co.T
        r2 = (d * d).sum(-1)
        ii, jj = torch.nonzero(r2 < want_list ** 2, as_tuple=True) if want_list else (torch.zeros(0), None)
        if want_list:
            entries += int((ii + r0 != jj).sum())
        ii, jj = torch.nonzero(r2 < rout0 ** 2, as_tuple=True)
        keep = jj > ii + r0
        ii, jj = ii[keep], jj[keep]
        for c0 in range(0, len(ii), 600000):
            a, j = ii[c0:c0 + 600000], jj[c0:c0 + 600000]
            rc, shift, rr = d[a, j], sh[a, j], torch.sqrt(r2[a, j])
            i = a + r0
            sw, dsw = torch.ones_like(rr), torch.zeros_like(rr)
            m = rr * rr >= rout * rout
            au, bu = (rout0 - 3.0 * rout + 2.0 * rr) / tol ** 3, rout0 - rr
            sw = torch.where(m, au * bu * bu, sw)
            dsw = torch.where(m, (-2.0 * au * bu + 2.0 * bu * bu / tol ** 3) / rr, dsw)
            tij = ss[g0[i]] + ss[g0[j]] - 2
            v = torch.zeros_like(rr)
            fs = zero3(len(rr))
            for u in range(kmax):
                for t in range(kmax):
                    has = (u < gn[i]) & (t < gn[j])
                    p = torch.nonzero(has).ravel()
                    if not len(p):
                        continue
                    ia, ib = g0[i[p]] + u, g0[j[p]] + t
                    ok = ~torch.isin(torch.minimum(ia, ib).add(1) * (n + 1) + torch.maximum(ia, ib).add(1), keys)
                    p, ia, ib = p[ok], ia[ok], ib[ok]
                    dx = (x[ia] - x[ib] - shift[p]) @ co.T
                    rsq = (dx * dx).sum(-1)
                    r = torch.sqrt(rsq)
                    erfc, ex2 = _erfc(s.alpha * r)
                    tw = 2.0 / math.sqrt(math.pi) * s.alpha * r * ex2
                    qq = q[ia] * q[ib]
                    if al is None:
                        k = lij[typ[ia], typ[ib]]
                        c12, c6 = e12[k], e6[k]
                        lj = c6 > 1e-12
                        i6 = 1.0 / rsq ** 3
                        conf = torch.where(lj, (c12 * i6 - c6) * i6, 0.0)
                        qf = torch.where(lj, (12.0 * c12 * i6 - 6.0 * c6) * i6 / rsq, 0.0)
                        cou = qq * erfc / r
                        qf = qf + qq * (erfc + tw) / (r * rsq)
                    else:
                        sa = ssa[ia] + ssa[ib]  # 2 plain, -1 with a removed atom, -4 both removed (or the added twins)

                        def factors(add, rem, sa=sa):
                            one = torch.where(sa == -1, rem, torch.where(sa == 3, add, 0.0))
                            two = torch.where(sa == 0, 0.0, 1.0 - one)
                            return one, two
                        ep = 4.0 * torch.sqrt(eps[ia] * eps[ib])
                        x6 = rsq ** 3 / (rmin[ia] + rmin[ib]) ** 6

                        def energy(l1, l2, q1, q2):
                            gp = al.ljsoft * l1 + x6
                            au2 = 1.0 / torch.sqrt(al.qsoft * q1 * q1 + rsq)
                            c = torch.where(ep > 1e-12, l2 * ep * (1.0 / gp ** 2 - 1.0 / gp), 0.0)
                            return gp, au2, c, q2 * qq * erfc * au2
                        l1, l2 = factors(ladd, lrm)
                        q1, q2 = factors(laddq, lrmq)
                        gp, au2, conf, cou = energy(l1, l2, q1, q2)
                        qf = torch.where(ep > 1e-12, 6.0 * x6 * l2 * ep * (2.0 / gp ** 3 - 1.0 / gp ** 2) / rsq, 0.0)
                        qf = qf + q2 * qq * au2 * (erfc * au2 * au2 + tw / rsq)
                        _, _, conf0, cou0 = energy(*factors(ladd0, lrm0), *factors(laddq0, lrmq0))
                        dw = dw + (sw[p] * (conf - conf0 + cou - cou0)).sum()
                    fv = (qf * sw[p])[:, None] * dx
                    f.index_add_(0, ia, fv)
                    f.index_add_(0, ib, -fv)
                    fs.index_add_(0, p, fv)
                    v.index_add_(0, p, conf + cou)
                    en.index_add_(0, tij[p], sw[p] * conf)
                    en.index_add_(0, tij[p] + 3, sw[p] * cou)
            x3 = -(dsw * v)[:, None] * rc
            for u in range(kmax):
                for grp, sign in ((i, 1.0), (j, -1.0)):
                    p = torch.nonzero(u < gn[grp]).ravel()
                    at = g0[grp[p]] + u
                    f.index_add_(0, at, sign * w[at][:, None] * x3[p])
            st -= (fs + x3).T @ shift
    st += f.T @ xm[mol]
    return f, en, st @ co.T, float(dw), entries, xm[mol]


def _spline(w, order):
    """Cardinal B-spline weights and their derivatives at fraction w (n,) -> (n, order)."""
    c = torch.zeros(len(w), order, dtype=torch.float64, device=w.device)
    c[:, 0], c[:, 1] = 1.0 - w, w

    def up(c, k):
        o = torch.zeros_like(c)
        for j in range(k):
            left = (w + (k - 1 - j)) * c[:, j - 1] if j else 0.0
            o[:, j] = (left + (1.0 + j - w) * c[:, j]) / (k - 1)
        return o
    for k in range(3, order):
        c = up(c, k)
    d = torch.zeros_like(c)
    d[:, 0] = -c[:, 0]
    d[:, 1:] = c[:, :-1] - c[:, 1:]
    return up(c, order), d


def _moduli(order, n):
    """Squared B-spline moduli with the single-precision 2 pi of the reference."""
    one, _ = _spline(torch.zeros(1, dtype=torch.float64), order)
    b = np.zeros(n + order)
    b[1:order + 1] = one[0].numpy()
    arg = 2.0 * _PI32 * np.outer(np.arange(n), np.arange(n)) / n
    m = (np.cos(arg) @ b[:n]) ** 2 + (np.sin(arg) @ b[:n]) ** 2
    for k in range(n):
        if m[k] < 1e-7:
            m[k] = 0.5 * (m[k - 1] + m[(k + 1) % n])
    return m


def _recip(s, q, dev, xmol, forces=True):
    """Smooth PME: energy, forces and the stress -vir + molecular correction."""
    K, p = s.nfft, s.order
    rec = 0.5 * np.array(s.oc).T                     # recip(i, j) = oc(j, i) / 2
    x = torch.stack([_t(c, dev) for c in (s.xp0, s.yp0, s.zp0)], 1)
    co = _t(np.array(s.co), dev)
    qd = _t(q, dev)
    fr = (x @ co.T) @ _t(rec, dev)
    fr = _t(np.array(K, float), dev) * (fr - torch.round(fr) + 0.5)
    b = fr.long()
    th, dt, idx = [], [], []
    for k in range(3):
        t, d = _spline(fr[:, k] - b[:, k], p)
        th.append(t)
        dt.append(d)
        idx.append((b[:, k:k + 1] - p + 1 + torch.arange(p, device=dev)) % K[k])
    flat = (idx[2][:, :, None, None] * K[1] + idx[1][:, None, :, None]) * K[0] + idx[0][:, None, None, :]
    val = th[2][:, :, None, None] * th[1][:, None, :, None] * th[0][:, None, None, :] * qd[:, None, None, None]
    grid = torch.zeros(K[0] * K[1] * K[2], dtype=torch.float64, device=dev).index_add_(0, flat.ravel(), val.ravel())
    F = np.fft.rfftn(grid.cpu().numpy().reshape(K[2], K[1], K[0]))
    H = K[0] // 2 + 1
    k1, k2, k3 = np.arange(H)[None, None, :], np.arange(K[1])[None, :, None], np.arange(K[2])[:, None, None]
    mm = [np.where(kk + 1 > (nk + 1) // 2, kk - nk, kk) for kk, nk in zip((k1, k2, k3), K)]
    h = [rec[a, 0] * mm[0] + rec[a, 1] * mm[1] + rec[a, 2] * mm[2] for a in range(3)]
    msq = h[0] ** 2 + h[1] ** 2 + h[2] ** 2
    msq[0, 0, 0] = 1.0
    fac = _PI32 ** 2 / s.alpha ** 2
    mod = [_moduli(p, nk) for nk in K]
    den = _PI32 * s.volume * mod[0][None, None, :H] * mod[1][None, :, None] * mod[2][:, None, None] * msq
    et = np.exp(-fac * msq) / den
    et[0, 0, 0] = 0.0
    vt = 2.0 * (fac * msq + 1.0) / msq
    edge = (k1 == 0) | ((k1 == H - 1) & (K[0] % 2 == 0))
    s2 = np.where(edge, 1.0, 2.0) * et * np.abs(F) ** 2
    # the reference's masks on the off-diagonal virial
    lo2, lo3 = k2 < H, k3 < H
    f12 = np.where(edge, 1.0, np.where((h[0] * h[1] < 0.0) & lo2, 0.0, 1.0))
    f13 = np.where(edge, 1.0, np.where((h[0] * h[2] < 0.0) & lo3, 0.0, 1.0))
    neg = h[1] * h[2] < 0.0
    f23 = np.where(edge, 1.0, np.where(lo2 == lo3, ~neg, neg).astype(float))
    vir = np.zeros((3, 3))
    for a in range(3):
        vir[a, a] = 0.5 * (s2 * (vt * h[a] * h[a] - 1.0)).sum()
    for a, c, m in ((0, 1, f12), (0, 2, f13), (1, 2, f23)):
        vir[a, c] = vir[c, a] = 0.5 * (s2 * vt * h[a] * h[c] * m).sum()
    # the m = 0 term adds nothing to the diagonal (s2 = 0 there)
    eer = 0.5 * s2.sum()
    if not forces:
        return eer, None, None
    et[0, 0, 0] = 1.0  # passed through unscaled, as the reference leaves it
    Q = _t(np.fft.irfftn(F * et, s=(K[2], K[1], K[0])) * (K[0] * K[1] * K[2]), dev).ravel()
    gq = Q[flat]
    fl = []
    for k, (w0, w1, w2) in enumerate(((dt[0], th[1], th[2]), (th[0], dt[1], th[2]), (th[0], th[1], dt[2]))):
        w = w2[:, :, None, None] * w1[:, None, :, None] * w0[:, None, None, :]
        fl.append(-K[k] * qd * (w * gq).sum((1, 2, 3)))
    f = torch.stack(fl, 1) @ _t(rec, dev).T
    corr = -(f.T @ ((x - xmol) @ co.T))
    return eer, f, corr.cpu().numpy() - vir


def _corrections(s, pairs, q, dev, factor=None, q0=None, factor0=None):
    """erf corrections of pairs (without image): forces, energy by class, energy on q0."""
    x = torch.stack([_t(c, dev) for c in (s.xp0, s.yp0, s.zp0)], 1) @ _t(np.array(s.co), dev).T
    ia, ib = (_t(pairs[k].astype(np.int64) - 1, dev) for k in range(2))
    d = x[ia] - x[ib]
    r = torch.sqrt((d * d).sum(-1))
    erfc, e2 = _erfc(s.alpha * r)
    erf = 1.0 - erfc
    q = _t(q, dev)
    qq = q[ia] * q[ib] * (1.0 if factor is None else _t(factor, dev))
    qf = -qq * (erf - 2.0 / math.sqrt(math.pi) * s.alpha * r * e2) / r ** 3
    f = torch.zeros(s.natoms, 3, dtype=torch.float64, device=dev)
    f.index_add_(0, ia, qf[:, None] * d)
    f.index_add_(0, ib, -qf[:, None] * d)
    cls = _t(s.ss_index.astype(np.int64) - 1, dev)[ia]
    e = torch.zeros(2, dtype=torch.float64, device=dev).index_add_(0, cls, -qq * erf / r)
    e0 = 0.0
    if q0 is not None:
        q0 = _t(q0, dev)
        qq0 = q0[ia] * q0[ib] * (1.0 if factor0 is None else _t(factor0, dev))
        e0 = float((-qq0 * erf / r).sum())
    return f, e.cpu().numpy(), e0


def _exact_system(s, dev, al=None, lam=None):
    """One resident evaluation: forces, energies, stress, list size (and the parts of dU/dlambda's step)."""
    f, en, st, dw, entries, xmol = _direct(s, dev, al, lam, want_list=s.rcut + s.rtol + s.rnei)
    qc = q0 = np.array(s.charge)
    if al is not None:
        qc = _scaled_charges(s.charge, al.ss_alchemy, lam[4], lam[5])
        q0 = _scaled_charges(s.charge, al.ss_alchemy, lam[6], lam[7])
    eer, fr, sr = _recip(s, qc, dev, xmol)
    f = f + fr
    st = st.cpu().numpy() + sr
    fc, ec, ec0 = _corrections(s, _corr_pairs(s), qc, dev, q0=q0 if al is not None else None)
    f = f + fc
    if al is not None and al.listqq is not None:
        def lq(add, rem):
            return np.where(al.ss_alchemy == 2, add, np.where(al.ss_alchemy == -2, -rem, 0.0))
        a, b = al.listqq[0] - 1, al.listqq[1] - 1

        def fac(v):
            return (1.0 - np.abs(v[a])) * (1.0 - np.abs(v[b])) - al.listqq[2]
        fq, eq, eq0 = _corrections(s, al.listqq, s.charge, dev, fac(lq(lam[4], lam[5])), s.charge,
                                   fac(lq(lam[6], lam[7])))
        f, ec, ec0 = f + fq, ec + eq, ec0 + eq0
    if al is None:
        qs = [float((s.charge[s.ss_index == c] ** 2).sum()) for c in (1, 2)]
        slf = [-v * s.alpha / math.sqrt(math.pi) for v in qs]
    else:
        slf = [-float((qc[s.ss_index == 1] ** 2).sum()) * s.alpha / math.sqrt(math.pi), 0.0]
    en = en.cpu().numpy()
    e = np.array([eer, en[0], en[2], en[1], en[3], en[5], en[4], ec[0], ec[1], slf[0], slf[1]])
    f = f.cpu().numpy()
    out = [[f[:, k].copy() for k in range(3)], dict(energies=e, stress=st, entries=entries)]
    if al is not None:
        eer0, _, _ = _recip(s, q0, dev, xmol, forces=False)
        self0 = -float((q0[s.ss_index == 1] ** 2).sum()) * s.alpha / math.sqrt(math.pi)
        parts = [dw, eer - eer0, float(ec.sum()) - ec0, slf[0] - self0]
        out.append([sum(parts)] + parts + [eer0])
    return out


def _scaled_charges(q, ss, add, rem):
    """(1 - |lambda|) q of the added and removed atoms."""
    lq = np.abs(np.where(ss == 2, add, np.where(ss == -2, rem, 0.0)))
    return np.where(lq == 1.0, 0.0, np.where(lq == 0.0, q, (1.0 - lq) * q))


def exact(case, seed):
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    kind = case["kind"]
    if kind == "md":
        return None
    if kind == "windows":
        s, al, states = _windows(case, seed)
        got = [_exact_system(s, dev, al, lam) for lam in states]
    else:
        systems = [_system(case, seed, k) for k in range(case["replicas"])]
        s = systems[0]
        if kind == "fft_pme":
            m = s.molecule_coms()
            eer, f, st = _recip(s, np.array(s.charge), dev, _t(m[:, s.atomp - 1].T, dev))
            f = f.cpu().numpy()
            return dict(f=[f[:, k].copy() for k in range(3)], eer=float(eer), stress=st)
        if kind == "direct":
            f, en, st, _, _, _ = _direct(s, dev)
            f, en = f.cpu().numpy(), en.cpu().numpy()
            return dict(f=[f[:, k].copy() for k in range(3)], energies=en[[0, 2, 1, 3, 5, 4]], stress=st.cpu().numpy(),
                        list=None)
        got = [_exact_system(s, dev) for s in systems]
    out = dict(f=[g[0] for g in got], system=[g[1] for g in got])
    if case["replicas"] > 8:
        e = out["system"]
        out["system"] = dict(energies=np.stack([v["energies"] for v in e]), stress=np.stack([v["stress"] for v in e]),
                             entries=np.array([v["entries"] for v in e]))
    if kind == "windows":
        out["dwrk"] = np.array([g[2] for g in got])
    return out
