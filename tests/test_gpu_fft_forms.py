"""The transforms where their mapping has edges: planes that just fit the LDS of
a workgroup and planes that just do not, odd and prime-power axes, every radix,
fewer rows than threads; FP64 against the oracle's fft_pme at the parity
tolerances, FP32 against FP64 (transforms of up to 2^14 points per plane: a few
times 6e-8 of the largest value)."""
import dataclasses

import numpy as np
import pytest

import oracle as O
from conftest import rel, relrms
from test_gpu_parity import E_TOL, F_TOL, _pme_gpu, _stress_close
from test_gpu_spread_forms import _random

pytestmark = pytest.mark.gpu

GRIDS = [(5, 5, 5), (6, 10, 8), (9, 7 + 1, 27), (25, 15, 12), (32, 32, 32), (27, 50, 6), (64, 48, 36), (45, 75, 16),
         (96, 96, 8), (100, 96, 8), (100, 100, 8), (128, 60, 10), (60, 128, 10), (16, 6, 120), (8, 5, 243)]


@pytest.mark.parametrize("nfft", GRIDS)
def test_grids(gpu_ctx, nfft):
    s = _random(n=300, nfft=nfft, order=4, L=30.0, seed=sum(nfft))
    g = _pme_gpu(gpu_ctx, s)
    o = O.fft_pme(s, variant="fftw")
    assert rel(g["eer"], o["eer"]) < E_TOL
    assert relrms(g["f"], o["f"]) < F_TOL
    assert _stress_close(g["stress"], o["stress"])


@pytest.mark.parametrize("nfft", [(20, 25, 18), (64, 64, 8), (128, 135, 8), (144, 144, 8)])
def test_fp32_and_batches(gpu_ctx, nfft):
    """FP32 planes, one plane form beside the other in a batch."""
    from orac_hip.api import Batch, ResidentSystem
    grids = [nfft, (100, 100, 8), (16, 16, 16)]
    f = []
    for precision in (0, 1):
        systems = [dataclasses.replace(_random(n=300, nfft=k, order=5, L=30.0, seed=9), rcut=8.0) for k in grids]
        # (no touching atoms: the reciprocal forces are what is compared)
        systems = [dataclasses.replace(s, ecc12=0.0 * s.ecc12, ecc6=0.0 * s.ecc6) for s in systems]
        rss = [ResidentSystem(gpu_ctx, s, precision=precision) for s in systems]
        alone = []
        for rs in rss:
            rs.eval(rebuild_list=True)
            alone.append(rs.results())
        b = Batch(gpu_ctx, rss)
        b.eval(rebuild_list=True)
        for r, a in zip(b.results(), alone):
            assert np.array_equal(r["f"], a["f"]) and r["eer"] == a["eer"]
        b.close()
        for rs in rss:
            rs.close()
        f.append(alone)
    for a, b in zip(*f):
        assert relrms(b["f"], a["f"]) < 2e-6 and rel(b["eer"], a["eer"]) < 2e-6
