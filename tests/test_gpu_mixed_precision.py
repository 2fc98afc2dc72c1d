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


@pytest.mark.parametrize("K,bound", [(72, 5.23e-7), (108, 7.55e-7)])
def test_reciprocal_forces_fp32(gpu_ctx, K, bound):
    """FP32 splines and transforms, mean of eight systems (every sum of a run is
    in fixed order).  The bounds lie between the error with the splines' sums
    fused and no twiddles inside radix 6 (5.07e-7, 7.34e-7) and with each product
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


@pytest.mark.parametrize("order", [0, 1])
def test_plain_system_beside_an_alchemical_one(gpu_ctx, order):
    """A plain system gets, in a launch with alchemical ones, what it gets alone."""
    from orac_hip.api import Batch, ResidentSystem
    for precision in (0, 1):
        s, a = grouped(sizes=[1, 3, 2]), grouped(sizes=[3], seed=5)
        rss = [ResidentSystem(gpu_ctx, x, precision=precision) for x in ([s, a] if order == 0 else [a, s])]
        k = rss[order]
        k.eval(rebuild_list=True)
        alone = k.results()
        rss[1 - order].set_alchemy(*_removed(a))
        rss[1 - order].eval(rebuild_list=True)
        window = rss[1 - order].results()
        b = Batch(gpu_ctx, rss)
        b.eval(rebuild_list=True)
        r = b.results()
        assert np.array_equal(r[order]["f"], alone["f"]) and r[order]["uconf_ss"] == alone["uconf_ss"]
        assert np.array_equal(r[1 - order]["f"], window["f"])
        b.close()
        for rs in rss:
            rs.close()
