"""The host-prepared tables and the index arithmetic the kernels share with the
host, compiled for the host (tests/host/probe.cpp) and checked without a GPU."""
import ctypes as C
import os
import subprocess

import numpy as np
import pytest

from conftest import PKG, ROOT


@pytest.fixture(scope="module")
def probe(tmp_path_factory):
    from orac_hip import build
    if not (os.path.exists(build.HIPCC) and os.path.exists(build.LIB)):
        pytest.skip("hipcc or liborac_hip.so not available")
    so = str(tmp_path_factory.mktemp("probe") / "probe.so")
    lib = os.path.join(PKG, "lib")
    subprocess.run([build.HIPCC, *build.HIP_FLAGS, "--cuda-host-only", "-shared", "-x", "hip",
                    os.path.join(ROOT, "tests", "host", "probe.cpp"), "-o", so, f"-L{lib}", "-lorac_hip",
                    f"-Wl,-rpath,{lib}"], check=True, capture_output=True)
    return C.CDLL(so)


def _ptr(a):
    return a.ctypes.data_as(C.c_void_p)


def _cell(a, b, c, alpha, beta, gamma):
    """co (half the cell vectors as columns) of lengths a, b, c and angles in degrees."""
    ca, cb, cg = np.cos(np.radians([alpha, beta, gamma]))
    sg = np.sqrt(1.0 - cg * cg)
    cy = (ca - cb * cg) / sg
    return 0.5 * np.array([[a, b * cg, c * cb], [0.0, b * sg, c * cy], [0.0, 0.0, c * np.sqrt(1.0 - cb * cb - cy * cy)]])


OCT = np.degrees(np.arccos(1.0 / 3.0))
# cell, cells per axis, list cutoff, whether some run along z does not reach dz = 0 and its neighbours
BOXES = {
    "cubic": (_cell(50, 50, 50, 90, 90, 90), (14, 14, 14), 10.0, False),
    "orthorhombic": (_cell(40, 55, 70, 90, 90, 90), (11, 15, 20), 10.6, False),
    "sheared_xy": (_cell(40, 40, 40, 90, 90, 65), (9, 9, 9), 6.0, False),
    "monoclinic": (_cell(50, 50, 50, 90, 120, 90), (14, 14, 14), 10.0, True),
    "sheared_yz": (_cell(50, 50, 50, 60, 90, 90), (14, 14, 14), 10.0, True),
    "octahedron": (_cell(45, 45, 45, OCT, 180.0 - OCT, OCT), (9, 9, 9), 9.5, True),
    "dodecahedron": (_cell(70, 70, 70, 60, 60, 90), (20, 20, 20), 11.0, True),
    "sixty": (_cell(45, 45, 45, 60, 60, 60), (19, 19, 19), 12.0, True),
    "uneven": (_cell(45, 60, 80, 60, 60, 90), (12, 17, 31), 10.0, True),
}


@pytest.mark.parametrize("name", list(BOXES))
def test_stencil_runs_are_the_stencil(probe, name):
    """The list build's runs along z visit, from every cell of a column, each of
    the stencil's cells once and stay inside the column."""
    from orac_hip.api import Context
    co, nc, rc, one_sided = BOXES[name]
    nind, ii, jj, kk = Context.lc_index(20000, *nc, rc, np.asfortranarray(co))
    n = int(nind[1])
    sten = np.ascontiguousarray(np.stack([v[1:2 * n:2] for v in (ii, jj, kk)], axis=1), np.int32)
    col = np.zeros((n, 4), np.int32)
    ncol = probe.probe_stencil_runs(_ptr(sten), n, _ptr(np.array(nc, np.int32)), _ptr(col))
    assert ncol > 0
    col = col[:ncol]
    assert bool(((col[:, 3] < -1) | (col[:, 2] > 1)).any()) == one_sided
    out = np.zeros(4, np.int32)
    for k in range(nc[2]):
        cells = []
        for dx, dy, z0, z1 in col.tolist():
            probe.probe_run_cells(k, z0, z1, nc[2], _ptr(out))
            a0, b0, a1, b1 = out.tolist()
            assert 0 <= a0 < b0 <= nc[2] and 0 <= a1 <= b1 <= nc[2]
            cells += [(dx, dy, z) for z in (*range(a0, b0), *range(a1, b1))]
        want = [(dx, dy, (k + dz) % nc[2]) for dx, dy, dz in sten.tolist()]
        assert sorted(cells) == sorted(want)


@pytest.mark.parametrize("smallest", [0, 1])
@pytest.mark.parametrize("order", [3, 4, 5, 6, 8])
@pytest.mark.parametrize("n,L,K", [(24000, 62.0, 64), (24000, 124.0, 96), (24000, 186.0, 144), (24000, 250.0, 160),
                                   (24000, 250.0, 200), (648, 18.6, 20), (648, 80.0, 64), (3, 40.0, 32)])
def test_spread_bins_hold_a_droplet(probe, n, L, K, order, smallest):
    """Every bin has room for a condensed phase (0.13 atoms per cubic A) wherever
    it lies in the box, and all bins together take no more than the grids or a
    fixed amount per atom and tile."""
    from math import ceil
    if not any(K % e == 0 for e in range(max(2, order - 1), 9)):
        pytest.skip("no tile edge")
    nbin = C.c_int()
    probe.probe_bin_cap.argtypes = [C.c_void_p, C.c_int, C.c_int, C.c_double, C.c_int, C.c_void_p]
    cap = probe.probe_bin_cap(_ptr(np.array([K] * 3, np.int32)), order, n, L ** 3, smallest, C.byref(nbin))
    assert cap >= min(n, ceil(0.13 * L ** 3 / nbin.value))
    assert cap * nbin.value <= max(2 * n + 48 * nbin.value, K ** 3)
