"""The tiled spread and the gather where their mapping has edges: bins that
overflow their slots (every atom in one corner), fewer atoms than a
wavefront, one tile along an axis, odd grids, every spline order; against the
oracle's fft_pme at the FP64 parity tolerances, and against the atomic spread
(integers on the grid: the same forces bit for bit)."""
import dataclasses

import numpy as np
import pytest

import oracle as O
from conftest import rel, relrms
from test_gpu_parity import E_TOL, F_TOL, _pme_gpu, _stress_close

pytestmark = pytest.mark.gpu


def _random(n, nfft, order, L=30.0, box=1.0, seed=2):
    """n free atoms (one group and molecule each) in the fraction `box` of the cell's edge."""
    from orac_hip import synth
    rng = np.random.default_rng(seed)
    x = rng.uniform(-box, box, (3, n)) - (1.0 - box)
    q = rng.normal(0, 0.5, n)
    half = L / 2
    i = np.arange(1, n + 1, dtype=np.int32)
    tt, e12, e6 = synth._lj_tables(np.array([2.0]), np.array([0.1]))
    return synth.System(
        L=L, xp0=x[0], yp0=x[1], zp0=x[2], charge=synth.charge_internal(q - q.mean()), mass=np.full(n, 12.0),
        nbtype=np.ones(n, np.int32), ntypes=1, type_table=tt, ecc12=e12, ecc6=e6,
        grppt=np.asfortranarray(np.stack([i, i])), atomg=i, atomp=i, ss_index=np.full(n, 2, np.int32),
        pmass=np.ones(n), co=np.asfortranarray(np.diag([half] * 3)), oc=np.asfortranarray(np.diag([1 / half] * 3)),
        volume=L ** 3, alpha=0.35, nfft=nfft, order=order, rcut=8.0)


CASES = {
    "orders3": dict(n=500, nfft=(24, 20, 30), order=3),
    "orders4": dict(n=500, nfft=(24, 20, 30), order=4),
    "orders5": dict(n=500, nfft=(24, 20, 30), order=5),
    "orders6": dict(n=500, nfft=(25, 30, 24), order=6),
    "orders7": dict(n=300, nfft=(24, 32, 40), order=7),
    "orders8": dict(n=300, nfft=(24, 32, 40), order=8),
    "one_tile": dict(n=40, nfft=(8, 16, 5), order=5),
    "few_atoms": dict(n=3, nfft=(20, 20, 20), order=5),
    "corner": dict(n=3000, nfft=(48, 48, 48), order=5, box=0.05),      # far beyond one bin's slots
    "half_full": dict(n=4000, nfft=(36, 40, 45), order=4, box=0.5),
}


@pytest.mark.parametrize("name", list(CASES))
def test_spread_and_gather(gpu_ctx, name, monkeypatch):
    s = _random(**CASES[name])
    g = _pme_gpu(gpu_ctx, s)
    o = O.fft_pme(s, variant="fftw")
    assert rel(g["eer"], o["eer"]) < E_TOL
    assert relrms(g["f"], o["f"]) < F_TOL
    assert _stress_close(g["stress"], o["stress"])
    again = _pme_gpu(gpu_ctx, s)  # (the bins are left empty for the next call)
    assert np.array_equal(again["f"], g["f"]) and again["eer"] == g["eer"]
    monkeypatch.setenv("ORAC_HIP_SPREAD_ATOMIC", "1")
    a = _pme_gpu(gpu_ctx, s)
    assert np.array_equal(a["f"], g["f"]) and a["eer"] == g["eer"]


def test_mixed_orders_in_one_batch(gpu_ctx):
    """Systems of different spline orders in one launch (the kernels with the
    order at run time) give each its forces alone, on every evaluation."""
    from orac_hip.api import Batch, ResidentSystem
    systems = [dataclasses.replace(_random(n=200, nfft=(20, 20, 20), order=p, L=24.0, seed=p), rcut=7.0)
               for p in (4, 5, 6, 8)]
    rss = [ResidentSystem(gpu_ctx, s) for s in systems]
    alone = []
    for rs in rss:
        rs.eval()
        alone.append(rs.results()["f"])
    b = Batch(gpu_ctx, rss)
    for graph in (False, True, True):
        b.eval(graph=graph)
        for r, a in zip(b.results(), alone):
            assert relrms(r["f"], a) < 1e-12
    b.close()
    for rs in rss:
        rs.close()
