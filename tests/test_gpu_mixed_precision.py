"""Mixed precision against FP64 of the same system, by term: what is exact by
construction (a pair's two forces, a system beside others), and how far the
FP32 pair arithmetic, splines and transforms are from 64 bits."""
import dataclasses

import numpy as np
import pytest

from conftest import relrms
from test_gpu_pair_forms import grouped

pytestmark = pytest.mark.gpu


def _eval(ctx, s, precision, alchemy=None):
    from orac_hip.api import ResidentSystem
    rs = ResidentSystem(ctx, s, precision=precision)
    if alchemy is not None:
        rs.set_alchemy(*alchemy)
    rs.eval(rebuild_list=True)
    r = rs.results()
    rs.close()
    return r


def _removed(s, n=40, lam=0.4):
    """Atoms 1..n of s being removed, at lambda lam."""
    from orac_hip import synth
    return synth.alchemy_for(s, np.arange(n)), synth.lambda_state(lam, lrm0=lam + 0.1)


def _direct(ctx, s, precision, alchemy=None):
    """The direct sum's forces: those beyond the same system's with a cutoff that no pair is within."""
    far = dataclasses.replace(s, rcut=0.5, rtol=0.01, rnei=0.01)
    return _eval(ctx, s, precision, alchemy)["f"] - _eval(ctx, far, precision, alchemy)["f"]


@pytest.mark.parametrize("alchemical", [False, True])
@pytest.mark.parametrize("charges", [False, True])
@pytest.mark.parametrize("name", ["waters", "mixed", "seven_one", "tails"])
def test_pair_forces_cancel(gpu_ctx, name, charges, alchemical):
    """Both sides of a pair round alike in FP32, so the direct forces sum to
    zero but for the FP64 sums (1,728 atoms of ~100 terms each: a few hundred
    roundings of 1e-16 of the largest; a single FP32 rounding is 6e-8)."""
    from test_gpu_pair_forms import CASES
    s = grouped(**CASES[name])
    if not charges:
        s = dataclasses.replace(s, charge=0.0 * s.charge)
    f = _direct(gpu_ctx, s, 1, _removed(s) if alchemical else None)
    assert np.abs(f.sum(axis=1)).max() < 1e-12 * np.abs(f).max()


def test_lj_energy_has_no_bias(gpu_ctx):
    """LJ constants that FP32 holds exactly: what is left of the energy's and
    the forces' error is the arithmetic's, whose roundings (6e-8 a pair) average
    out over 100,000 pairs unless a seed's bias is raised to the twelfth power
    (1.4e-7 of the energy where r^-6 came from the reciprocal square root)."""
    s = grouped(sizes=[3])
    s = dataclasses.replace(s, charge=0.0 * s.charge, ecc12=np.exp2(np.round(np.log2(s.ecc12.clip(1e-300)))) * (s.ecc12 > 0),
                            ecc6=np.exp2(np.round(np.log2(s.ecc6.clip(1e-300)))) * (s.ecc6 > 0))
    g, m = _eval(gpu_ctx, s, 0), _eval(gpu_ctx, s, 1)
    e, em = (sum(r[k] for k in ("uconf_slt", "uconf_slv", "uconf_ss")) for r in (g, m))
    tr, trm = (np.trace(r["stress"]) for r in (g, m))
    print("LJ energy", (em - e) / abs(e), "stress", (trm - tr) / abs(tr), "f", relrms(m["f"], g["f"]))
    # (energy: a sum of both signs; 1.1e-7 and 2.4e-8 here, 8.7e-7 and 2.1e-7 with the seed's powers)
    assert abs(em - e) < 2e-7 * abs(e)
    assert abs(trm - tr) < 6e-8 * abs(tr)


@pytest.mark.parametrize("K,bound", [(72, 5.23e-7), (108, 7.55e-7)])
def test_reciprocal_forces_fp32(gpu_ctx, K, bound):
    """FP32 splines and transforms, mean of eight systems (every sum of a run is
    in fixed order).  The bounds lie between the error with the splines' sums
    fused and no twiddles inside radix 6 (5.07e-7, 7.34e-7; 4.95e-7, 7.28e-7 with
    the moduli of the rounded splines and transforms) and with each product
    rounded and radix 6 as 2 x 3 (5.39e-7, 7.75e-7)."""
    err = []
    for seed in range(8):
        s = grouped(sizes=[1], side=20, spacing=K / 20.0, seed=seed)
        s = dataclasses.replace(s, nfft=(K, K, K), order=5, rcut=0.3, rtol=0.01, rnei=0.01, ecc12=0 * s.ecc12,
                                ecc6=0 * s.ecc6)
        g, m = _eval(gpu_ctx, s, 0), _eval(gpu_ctx, s, 1)
        err.append(relrms(m["f"], g["f"]))
    print("reciprocal", K, np.mean(err), err)
    assert np.mean(err) < bound


def _reciprocal_energy(ctx, K, order):
    """Relative error of the FP32 reciprocal energy, mean of eight systems."""
    err = []
    for seed in range(8):
        s = grouped(sizes=[1], side=12, spacing=K / 12.0, seed=seed)
        s = dataclasses.replace(s, nfft=(K, K, K), order=order, rcut=0.3, rtol=0.01, rnei=0.01, ecc12=0 * s.ecc12,
                                ecc6=0 * s.ecc6)
        g, m = _eval(ctx, s, 0), _eval(ctx, s, 1)
        err.append((m["eer"] - g["eer"]) / abs(g["eer"]))
    print("reciprocal energy", K, order, np.mean(err), err)
    return np.mean(err)


@pytest.mark.parametrize("order", [4, 5, 6, 7, 8])
def test_reciprocal_energy_has_the_splines_charge(gpu_ctx, order):
    """The factors 1/3, 1/5, ... of the splines' recurrence, rounded, scale every
    weight of an axis alike, and the energy by their sixth power (order 5: 1.8e-7;
    6: 2.7e-7): the moduli take it out.  What is left is below two roundings, 1.2e-7
    (3.5e-8 to 4.3e-8 measured; 2.1e-7 to 7.6e-7 with the exact splines' moduli; 0.4e-8
    to 1.2e-8 where the transforms' gain is taken out too)."""
    assert abs(_reciprocal_energy(gpu_ctx, 40, order)) < 2.0 ** -23


@pytest.mark.parametrize("K", [24, 32, 36, 48, 54, 72, 80, 96])
def test_reciprocal_energy_fp32(gpu_ctx, K):
    """Grids of every radix: the rounding of the transforms' constants (sqrt(3/4),
    cos(2 pi / 5), ...) and twiddle factors scales a mode, and the moduli carry
    that.  The mean error is at most 3.6e-8 (a system's deviation of 1 to 3e-8 is
    the rounding of the arithmetic), and 7.6e-8 to 1.0e-7 without; the bound is one
    rounding, 2^-24."""
    assert abs(_reciprocal_energy(gpu_ctx, K, 5)) < 2.0 ** -24


@pytest.mark.parametrize("beside", ["alchemical", "two_shells"])
@pytest.mark.parametrize("order", [0, 1])
def test_plain_system_beside_another(gpu_ctx, order, beside):
    """A plain system gets, in a launch with alchemical ones or with outer shells
    that skip the Ewald term, what it gets alone; so does the other."""
    from orac_hip.api import Batch, ResidentSystem
    for precision in (0, 1):
        s, a = grouped(sizes=[1, 3, 2]), grouped(sizes=[3], seed=5)
        rss = [ResidentSystem(gpu_ctx, x, precision=precision) for x in ([s, a] if order == 0 else [a, s])]
        k, other = rss[order], rss[1 - order]
        k.eval(rebuild_list=True)
        alone = k.results()
        if beside == "alchemical":
            other.set_alchemy(*_removed(a))
        else:
            other.set_shells(4.5, 0.5)
        other.eval(rebuild_list=True)
        want = other.results()
        b = Batch(gpu_ctx, rss)
        b.eval(rebuild_list=True)
        r = b.results()
        assert np.array_equal(r[order]["f"], alone["f"]) and r[order]["uconf_ss"] == alone["uconf_ss"]
        assert np.array_equal(r[1 - order]["f"], want["f"])
        b.close()
        for rs in rss:
            rs.close()


def test_window_against_fp64(gpu_ctx):
    """Windows of a ligand being removed: forces, stress and the energy step to
    the next window, whose terms nearly cancel."""
    from orac_hip import api, synth
    s, al, states = synth.alchemy_windows(n_windows=6, seed=41)
    out = []
    for precision in (0, 1):
        f, st, dw = [], [], []
        for lam in states:
            rs = api.ResidentSystem(gpu_ctx, s, precision=precision)
            rs.set_alchemy(al, lam)
            rs.eval(rebuild_list=True)
            r = rs.results()
            f.append(r["f"])
            st.append(r["stress"])
            dw.append(rs.alchemy_results()["dwrk"])
            rs.close()
        out.append((np.array(f), np.array(st), np.array(dw)))
    # (stress 3.4e-8; 1.9e-7 where a pair's two sides round apart and LJ takes the seed's powers)
    assert relrms(out[1][1], out[0][1]) < 8e-8
    print("windows f", relrms(out[1][0], out[0][0]), "stress", relrms(out[1][1], out[0][1]), "dwrk", out[0][2],
          np.abs(out[1][2] - out[0][2]).max())
