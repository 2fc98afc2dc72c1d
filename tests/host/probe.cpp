// Host-side pieces of the library for the tests that run without a GPU: the
// same inline functions the kernels call, and the tables the host prepares.
#include "../../orac-porting_amd/csrc/host.hpp"

using namespace orac;

// col[4 * ncol]: the stencil's runs along z; returns ncol
extern "C" int probe_stencil_runs(const int *sten, int nsten, const int *nc, int *col) {
  const std::vector<int4> r = stencil_runs(std::vector<int>(sten, sten + 3 * (size_t)nsten), nc[0], nc[1], nc[2]);
  for (size_t k = 0; k < r.size(); ++k) {
    const int v[4] = {r[k].x, r[k].y, r[k].z, r[k].w};
    std::copy(v, v + 4, col + 4 * k);
  }
  return (int)r.size();
}

// out[4]: the run's cells as [a0, b0) and [a1, b1)
extern "C" void probe_run_cells(int k, int z0, int z1, int n, int *out) {
  const RunCells r = run_cells(k, z0, z1, n);
  const int v[4] = {r.a0, r.b0, r.a1, r.b1};
  std::copy(v, v + 4, out);
}

// room of one spread bin, and the tiles, for the largest or smallest tiles
extern "C" int probe_bin_cap(const int *K, int order, int natoms, double volume, int smallest, int *nbin) {
  PmeDesc d;
  std::memset(&d, 0, sizeof d);
  d.K1 = K[0];
  d.K2 = K[1];
  d.K3 = K[2];
  d.order = order;
  d.natoms = natoms;
  d.volume = volume;
  pme_tiling(d, smallest != 0);
  *nbin = d.nb1 * d.nb2 * d.nb3;
  return d.bin_cap;
}
