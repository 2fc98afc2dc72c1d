"""The resident list build where its mapping has edges: one crowded cell,
cells of more members than a wavefront has lanes, the smallest grids whose
stencil does not fold, runs that wrap at either face of the box or lie wholly
past it (cells whose third vector leans on the others), every cell count in
between; the entries are exactly the ordered pairs within
the cutoff, and the forces the oracle's at the FP64 parity tolerances."""
import dataclasses

import numpy as np
import pytest

import oracle as O
from conftest import relrms
from test_gpu_parity import F_TOL
from test_gpu_spread_forms import _random
from test_host_tables import OCT, _cell

pytestmark = pytest.mark.gpu

CASES = {
    "one_cell": dict(n=700, ncell=1),
    "folds": dict(n=300, ncell=3),          # the stencil would fold: built as one cell
    "smallest": dict(n=500, ncell=7, L=30.0),
    "odd": dict(n=900, ncell=9),
    "many": dict(n=400, ncell=17),          # more cells than groups, some of them empty
    "crowded": dict(n=1500, ncell=9, box=0.12),   # > 64 members in a cell
    "faces": dict(n=600, ncell=8, box=0.3, shift=-0.3),  # members across all three faces
    "sheared_xy": dict(n=800, ncell=9, skew=0.3),
    # runs along z that do not reach the owner's own layer or the next one
    "monoclinic": dict(n=900, ncell=14, cell=_cell(30, 30, 30, 90, 120, 90)),
    "sheared_yz": dict(n=900, ncell=14, cell=_cell(30, 30, 30, 60, 90, 90)),
    "octahedron": dict(n=800, ncell=9, cell=_cell(28.4, 28.4, 28.4, OCT, 180.0 - OCT, OCT)),
    "dodecahedron": dict(n=1200, ncell=20, cell=_cell(38, 38, 38, 60, 60, 90)),
    "sixty": dict(n=700, ncell=19, cell=_cell(24, 24, 24, 60, 60, 60)),
    "few": dict(n=3, ncell=8),
    "scan_rows": dict(n=300, ncell=16),     # one cell past the scan's rows of 4,096
    "scan_rounds": dict(n=300, ncell=27),   # more cells than one round of the scan
}


@pytest.mark.parametrize("cell_order", [0, 1])
@pytest.mark.parametrize("name", list(CASES))
def test_list_build(gpu_ctx, name, cell_order):
    from orac_hip.api import Batch, Context, ResidentSystem
    c = dict(CASES[name])
    ncell, shift, skew, cell = c.pop("ncell"), c.pop("shift", 0.0), c.pop("skew", 0.0), c.pop("cell", None)
    s = _random(nfft=(24, 24, 24), order=4, **c)
    co = np.array(s.co) if cell is None else np.array(cell)
    co[0, 1] += skew * co[0, 0]
    s = dataclasses.replace(s, volume=8.0 * np.linalg.det(co))
    wrap = lambda x: (x + shift + 1.0) % 2.0 - 1.0
    # no Lennard-Jones terms: a few touching atoms would hide every other pair's force
    s = dataclasses.replace(s, rcut=5.0, rtol=0.3, rnei=0.7, co=np.asfortranarray(co), ecc12=0.0 * s.ecc12,
                            ecc6=0.0 * s.ecc6,
                            oc=np.asfortranarray(np.linalg.inv(co)), xp0=wrap(s.xp0), yp0=wrap(s.yp0), zp0=wrap(s.zp0))
    x = np.stack([s.xp0, s.yp0, s.zp0])
    d = x[:, :, None] - x[:, None, :]
    d -= 2.0 * np.round(0.5 * d)
    r2 = ((np.einsum("ij,jkl->ikl", co, d)) ** 2).sum(0)
    cut = (s.rcut + s.rtol + s.rnei) ** 2
    assert np.abs(r2 / cut - 1.0).min() > 1e-9  # (no pair within rounding of the cutoff)
    pairs = int((r2 < cut).sum()) - s.natoms
    if cell is not None:
        nind, ii, jj, kk = Context.lc_index(20000, ncell, ncell, ncell, cut ** 0.5, np.asfortranarray(co))
        runs = {}
        for dx, dy, dz in zip(*(v[1:2 * nind[1]:2].tolist() for v in (ii, jj, kk))):
            runs.setdefault((dx, dy), []).append(dz)
        assert any(max(z) < -1 or min(z) > 1 for z in runs.values())
    rs = ResidentSystem(gpu_ctx, s, precision=0, ncell=ncell)
    b = Batch(gpu_ctx, [rs])
    b.set_tuning(cell_order=cell_order)
    b.eval(rebuild_list=True)
    g = b.results()[0]
    b.eval(rebuild_list=True)
    assert np.array_equal(b.results()[0]["f"], g["f"])
    b.close()
    rs.close()
    assert g["list_entries"] == pairs
    fa = O.ForceArgs(s)
    half = [np.flatnonzero(r2[i, :i] < cut) + 1 for i in range(s.natoms)]
    nnlpp = np.concatenate([np.concatenate([[len(h)], h]) for h in half]).astype(np.int32)
    o = O.force(s, nnlpp, fa=fa, rinn=0.0, rout=s.rcut, rtolinn=0.0, rtolout=s.rtol, rneigh=0.0)
    f = o["f"] + O.fft_pme(s, variant="fftw")["f"]
    assert relrms(g["f"], f) < F_TOL


@pytest.mark.parametrize("sizes", [[1], [2, 4], [3, 5, 8], [16, 1, 17], [64, 7, 4]])
def test_prepare_group_and_molecule_sizes(gpu_ctx, sizes):
    """Centres, records and bins of groups (molecules, too) around the four
    lanes that share one and around MOL_SMALL atoms: forces and the virial,
    whose molecular correction reads the molecules' centres, against the oracle."""
    from orac_hip.api import ResidentSystem
    from test_gpu_pair_forms import grouped
    from test_gpu_parity import _stress_close
    from test_gpu_resident import oracle_total
    s = grouped(sizes)
    none = np.zeros((2, 0), np.int32)
    rs = ResidentSystem(gpu_ctx, s, precision=0)
    rs.eval(rebuild_list=True)
    g = rs.results()
    rs.close()
    o = oracle_total(s, none, np.zeros(0))
    assert relrms(g["f"], o["f"]) < F_TOL
    assert _stress_close(g["stress"], o["stress"])
