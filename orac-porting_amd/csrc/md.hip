// md.hip -- on-device r-RESPA integration of resident systems on gfx950.
//
// Two time levels of ORAC's multiple-time-step integrator (mtsmd.f), in its
// order of operations: the fast level (ORAC's n0 level: the solute's
// intramolecular harmonic distance terms) runs ninner substeps of
// h = dt/ninner inside one step dt of the slow level (ORAC's m level: the full
// nonbonded force -- direct space, PME, corrections -- with a single shell).
// Rigid units (3-site waters) are constrained by ORAC's matrix-inversion
// SHAKE after every drift and its RATTLE after every kick:
//
//   v += Fs*0.5*dt/m; RATTLE                                 (:2598-2604)
//   ninner times:  x += h*v + Ff*0.5*h^2/m; v += Ff*0.5*h/m;
//                  SHAKE against the positions before        (:2663-2683)
//                  Ff(x); v += Ff*0.5*h/m; RATTLE            (:2843-2884)
//   Fs(x)          (the force evaluation of the engine)
//   v += Fs*0.5*dt/m; RATTLE                                 (:3121-3146)
//
// A unit without harmonic terms moves alone between two slow forces, and an
// atom with terms moves with the atoms its terms reach, so the whole fast level
// of a step is one launch (k_md_advance): the units' kicks and substeps stay in
// registers, the atoms that terms connect share a workgroup.  It also closes
// the step before it.
//
// Positions are Cartesian FP64 with the reduced copy xp = oc x refreshed after
// every drift; the force path reads the reduced copy.  A unit is one atom or
// one rigid 3-atom molecule; one thread advances a unit, so constraint
// iterations stay in registers.  Every reduction (kinetic and bond energy) is
// per system and in fixed order.
#include <algorithm>

#include "common.hpp"
#include "kernels.hpp"

namespace orac {

__device__ inline void to_reduced(const double *oc, double x, double y, double z, double &xp, double &yp, double &zp) {
  xp = oc[0] * x + oc[3] * y + oc[6] * z;
  yp = oc[1] * x + oc[4] * y + oc[7] * z;
  zp = oc[2] * x + oc[5] * y + oc[8] * z;
}

// Constraints of one rigid triangle by ORAC's matrix-inversion method (MIM),
// the branch ORAC takes for molecules of at most mim_lim constraints
// (default 20, blkdta.f90:361): SHAKE after a drift as rattle_verlet.f:228-560
// does it, RATTLE after a kick as rattle_correc.f:176-385.  Constraint order
// (0,1), (0,2), (1,2); im = 1/m; dss the squared lengths.  mim_dir gives the
// direction in which atom `at` moves for constraint (ca, cb) with bond vector
// d (rattle_verlet.f:286-303): -d for its first atom, +d for its second.
// That is mim_sgn times d; its zeros are left out of the sums below (a third of
// their terms), which changes no value.
constexpr int MIM_CA[3] = {0, 0, 1}, MIM_CB[3] = {1, 2, 2};
__device__ constexpr int mim_sgn(int at, int k) {
  return at == (k == 2 ? 1 : 0) ? -1 : (at == (k == 0 ? 1 : 2) ? 1 : 0);
}
__device__ inline double3 mim_fma(double c, double3 d, double3 s) {
  return make_double3(s.x + d.x * c, s.y + d.y * c, s.z + d.z * c);
}
__device__ inline double mim_dot(double3 a, double3 b) { return a.x * b.x + a.y * b.y + a.z * b.z; }
__device__ inline double3 mim_diff(double3 a, double3 b) { return make_double3(a.x - b.x, a.y - b.y, a.z - b.z); }

// one element of the constraint matrix: (direction of ka's atoms for kb) . x, by inverse masses
__device__ inline double mim_elem(int ka, int kb, double dot, const double (&im)[3]) {
  const int sa = mim_sgn(MIM_CA[ka], kb), sb = mim_sgn(MIM_CB[ka], kb);
  if (sa && sb) return dot * im[MIM_CA[ka]] + dot * im[MIM_CB[ka]];
  return sa ? -sa * dot * im[MIM_CA[ka]] : sb * dot * im[MIM_CB[ka]];
}

// 3x3 solve by cofactors (rattle_verlet.f:381-397); later solves reuse them
struct MimInv {
  double b11, b12, b13, b21, b22, b23, b31, b32, b33, det;
};

__device__ inline MimInv mim_inverse(const double (&m)[3][3]) {
  MimInv r;
  const double a11 = m[0][0], a12 = m[0][1], a13 = m[0][2], a21 = m[1][0], a22 = m[1][1], a23 = m[1][2],
               a31 = m[2][0], a32 = m[2][1], a33 = m[2][2];
  r.b11 = a22 * a33 - a32 * a23;
  r.b12 = -a21 * a33 + a31 * a23;
  r.b13 = a21 * a32 - a22 * a31;
  r.b21 = -a12 * a33 + a32 * a13;
  r.b22 = a11 * a33 - a31 * a13;
  r.b23 = -a11 * a32 + a31 * a12;
  r.b31 = a12 * a23 - a22 * a13;
  r.b32 = -a11 * a23 + a21 * a13;
  r.b33 = a11 * a22 - a21 * a12;
  r.det = 1.0 / (a11 * r.b11 + a21 * r.b21 + a31 * r.b31);
  return r;
}

__device__ inline void mim_solve(const MimInv &r, double (&g)[3]) {
  const double xd = r.b11 * g[0] + r.b21 * g[1] + r.b31 * g[2];
  const double yd = r.b12 * g[0] + r.b22 * g[1] + r.b32 * g[2];
  const double zd = r.b13 * g[0] + r.b23 * g[1] + r.b33 * g[2];
  g[0] = xd * r.det;
  g[1] = yd * r.det;
  g[2] = zd * r.det;
}

constexpr double MIM_TOL = 1.0e-7;  // relative change of the multipliers (rattle_verlet.f:77)
constexpr int MIM_MAXIT = 120;      // rattle_verlet.f:461

// SHAKE: q are the drifted positions, p the positions before the drift (whose
// bond vectors give the directions of the corrections); v += correction * dti.
// The multipliers solve dss = |q_ij + corrections|^2 by iterating on the
// quadratic term; that term weights every constraint with the masses of the
// last constraint's atoms, as rattle_verlet.f:406-407 does.  Returns false
// when MIM_MAXIT iterations do not converge (the reference then starts the
// molecule over; here the unit is counted as failed and keeps what it has).
__device__ inline bool shake_mim3(double3 (&q)[3], const double3 (&p)[3], const double (&im)[3], const double *dss,
                                  double dti, double3 (&v)[3]) {
  double3 x0[3], xc[3];
  double dd[3], mat[3][3];
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    x0[k] = mim_diff(p[MIM_CA[k]], p[MIM_CB[k]]);
    xc[k] = mim_diff(q[MIM_CA[k]], q[MIM_CB[k]]);
  }
#pragma unroll
  for (int ka = 0; ka < 3; ++ka) {
    dd[ka] = dss[ka] - mim_dot(xc[ka], xc[ka]);
#pragma unroll
    for (int kb = 0; kb < 3; ++kb) mat[ka][kb] = -(mim_elem(ka, kb, mim_dot(x0[kb], xc[ka]), im) * 4.0);
  }
  const MimInv inv = mim_inverse(mat);
  const double gg1 = im[MIM_CA[2]] * 2.0, gg2 = im[MIM_CB[2]] * 2.0;  // the last constraint's atoms
  double gam[3] = {0.0, 0.0, 0.0};
  bool ok = true;
  for (int iter = 0;;) {
    const double gamo[3] = {gam[0], gam[1], gam[2]};
    double g[3];
#pragma unroll
    for (int ka = 0; ka < 3; ++ka) {
      double3 s = make_double3(0.0, 0.0, 0.0);
      if (iter > 0) {
#pragma unroll
        for (int kb = 0; kb < 3; ++kb) {
          const int sa = mim_sgn(MIM_CA[ka], kb), sb = mim_sgn(MIM_CB[ka], kb);
          if (sa) s = mim_fma(sa * (gam[kb] * gg1), x0[kb], s);
          if (sb) s = mim_fma(-sb * (gam[kb] * gg2), x0[kb], s);
        }
      }
      g[ka] = dd[ka] - mim_dot(s, s);
    }
    mim_solve(inv, g);
#pragma unroll
    for (int ka = 0; ka < 3; ++ka) gam[ka] = g[ka];
    ++iter;
    if (iter > MIM_MAXIT) {
      ok = false;
      break;
    }
    bool more = false;
#pragma unroll
    for (int ka = 0; ka < 3; ++ka)
      if (gam[ka] != 0.0 && fabs(gam[ka] - gamo[ka]) > MIM_TOL * fabs(gam[ka])) more = true;
    if (!more) break;
  }
  // corrections, each atom once: by the first constraint that holds it
  // (rattle_verlet.f:514-541)
#pragma unroll
  for (int at = 0; at < 3; ++at) {
    const double w = im[at] * 2.0;
#pragma unroll
    for (int kb = 0; kb < 3; ++kb) {
      const int s = mim_sgn(at, kb);
      if (!s) continue;
      const double aux = s * (gam[kb] * w);
      q[at] = mim_fma(aux, x0[kb], q[at]);
      v[at] = mim_fma(aux * dti, x0[kb], v[at]);
    }
  }
  return ok;
}

// RATTLE: velocities made orthogonal to the bonds at positions r by one
// linear solve (rattle_correc.f:176-385).
__device__ inline void rattle_mim3(const double3 (&r)[3], double3 (&v)[3], const double (&im)[3]) {
  double3 bv[3];
  double mat[3][3], gam[3];
#pragma unroll
  for (int k = 0; k < 3; ++k) bv[k] = mim_diff(r[MIM_CA[k]], r[MIM_CB[k]]);
#pragma unroll
  for (int ka = 0; ka < 3; ++ka) {
    gam[ka] = -mim_dot(mim_diff(v[MIM_CA[ka]], v[MIM_CB[ka]]), bv[ka]);
#pragma unroll
    for (int kb = 0; kb < 3; ++kb) mat[ka][kb] = -(mim_elem(ka, kb, mim_dot(bv[ka], bv[kb]), im) * 2.0);
  }
  mim_solve(mim_inverse(mat), gam);
#pragma unroll
  for (int at = 0; at < 3; ++at) {
    const double w = im[at] * 2.0;
#pragma unroll
    for (int kb = 0; kb < 3; ++kb) {
      const int s = mim_sgn(at, kb);
      if (!s) continue;
      v[at].x = v[at].x + (bv[kb].x * (s * gam[kb])) * w;
      v[at].y = v[at].y + (bv[kb].y * (s * gam[kb])) * w;
      v[at].z = v[at].z + (bv[kb].z * (s * gam[kb])) * w;
    }
  }
}

// v += f*0.5*dt/m, then RATTLE of a rigid unit (correc + rattle_correc): verlet.f's and correc.f's association
template <int NA>
__device__ __forceinline__ void md_kick(const double *fx, const double *fy, const double *fz, int a0, double dt,
                                        const double3 (&x)[NA], double3 (&v)[NA], const double (&m)[NA],
                                        const double (&im)[NA]) {
#pragma unroll
  for (int k = 0; k < NA; ++k) {
    v[k].x = v[k].x + gmem(fx)[a0 + k] * 0.5 * dt / m[k];
    v[k].y = v[k].y + gmem(fy)[a0 + k] * 0.5 * dt / m[k];
    v[k].z = v[k].z + gmem(fz)[a0 + k] * 0.5 * dt / m[k];
  }
  if constexpr (NA == 3) rattle_mim3(x, v, im);
}

// the kicks that end a step and those that start the next, in mtsmd.f's order
template <int NA>
__device__ __forceinline__ void md_kicks(const MdDesc &d, int a0, double dt, double hm, int flags,
                                         const double3 (&x)[NA], double3 (&v)[NA], const double (&m)[NA],
                                         const double (&im)[NA]) {
  if (flags & MD_END_MID) md_kick<NA>(d.fmx, d.fmy, d.fmz, a0, hm, x, v, m, im);
  if (flags & MD_END_SLOW) md_kick<NA>(d.fx, d.fy, d.fz, a0, dt, x, v, m, im);
  if (flags & MD_KICK_SLOW) md_kick<NA>(d.fx, d.fy, d.fz, a0, dt, x, v, m, im);
  if (flags & MD_KICK_MID) md_kick<NA>(d.fmx, d.fmy, d.fmz, a0, hm, x, v, m, im);
}

template <int NA>
__device__ __forceinline__ void md_load(const MdDesc &d, int a0, double3 (&x)[NA], double3 (&v)[NA], double (&m)[NA],
                                        double (&im)[NA]) {
#pragma unroll
  for (int k = 0; k < NA; ++k) {
    const int a = a0 + k;
    m[k] = gmem(d.mass)[a];
    im[k] = 1.0 / m[k];
    x[k] = make_double3(gmem(d.x)[a], gmem(d.y)[a], gmem(d.z)[a]);
    v[k] = make_double3(gmem(d.vx)[a], gmem(d.vy)[a], gmem(d.vz)[a]);
  }
}

__device__ __forceinline__ void md_store_v(const MdDesc &d, int a, double3 v) {
  gmem(d.vx)[a] = v.x;
  gmem(d.vy)[a] = v.y;
  gmem(d.vz)[a] = v.z;
}

__device__ __forceinline__ void md_store_x(const MdDesc &d, int a, double3 x) {
  gmem(d.x)[a] = x.x;
  gmem(d.y)[a] = x.y;
  gmem(d.z)[a] = x.z;
  double xp, yp, zp;
  to_reduced(d.oc, x.x, x.y, x.z, xp, yp, zp);
  gmem(d.xp)[a] = xp;
  gmem(d.yp)[a] = yp;
  gmem(d.zp)[a] = zp;
}

// a stage between two steps of one run: past the run's last step only what ends that step is left
__device__ inline int md_stage(const MdDesc &d, int flags) {
  if ((flags & MD_BETWEEN) && gmem(d.step)[0] == gmem(d.step)[1]) flags &= MD_END_MID | MD_END_SLOW;
  return flags;
}

// One unit's share of an integration stage, in ORAC's order (mtsmd.f):
//   MD_KICK_FAST  v += Ff*0.5*h/m, RATTLE        correc + rattle_correc (:2876-2884)
//   MD_END_MID    v += Fm*0.5*hm/m, RATTLE       the inner nonbonded shell (two shells)
//   MD_END_SLOW   v += Fs*0.5*dt/m, RATTLE       correc + rattle_correc (:3121-3146)
//   MD_KICK_SLOW, MD_KICK_MID                    the same kicks, starting the next step (:2598-2604)
//   MD_VERLET     x += h*v + Ff*0.5*h^2/m, v += Ff*0.5*h/m, then SHAKE against the
//                 positions before the drift      verlet + rattle_verlet (:2663-2683)
//   MD_RATTLE     RATTLE alone
// applied in that order when several are set.  Ff are the fast forces, Fs the
// slow ones.  One thread per unit; NA atoms per unit as a template parameter
// so the unit stays in registers.
template <int NA>
__device__ __forceinline__ void md_unit(const MdDesc &d, int u, int a0, double dt, double hm, double h, int flags) {
  double3 x[NA], v[NA];
  double m[NA], im[NA];
  md_load<NA>(d, a0, x, v, m, im);
  if (flags & MD_KICK_FAST) md_kick<NA>(d.bfx, d.bfy, d.bfz, a0, h, x, v, m, im);
  md_kicks<NA>(d, a0, dt, hm, flags, x, v, m, im);
  if (flags & MD_VERLET) {
    double3 p[NA];
    const double ts2 = h * h;
#pragma unroll
    for (int k = 0; k < NA; ++k) {
      const double3 f = make_double3(gmem(d.bfx)[a0 + k], gmem(d.bfy)[a0 + k], gmem(d.bfz)[a0 + k]);
      p[k] = x[k];
      x[k].x = x[k].x + h * v[k].x + f.x * 0.5 * ts2 / m[k];
      x[k].y = x[k].y + h * v[k].y + f.y * 0.5 * ts2 / m[k];
      x[k].z = x[k].z + h * v[k].z + f.z * 0.5 * ts2 / m[k];
      v[k].x = v[k].x + f.x * 0.5 * h / m[k];
      v[k].y = v[k].y + f.y * 0.5 * h / m[k];
      v[k].z = v[k].z + f.z * 0.5 * h / m[k];
    }
    if constexpr (NA == 3)
      if (!shake_mim3(x, p, im, d.ud2 + 3 * (size_t)u, h != 0.0 ? 1.0 / h : 0.0, v)) atomicAdd(d.fail, 1);
  }
  if constexpr (NA == 3)
    if (flags & MD_RATTLE) rattle_mim3(x, v, im);
#pragma unroll
  for (int k = 0; k < NA; ++k) {
    md_store_v(d, a0 + k, v[k]);
    if (flags & MD_VERLET) md_store_x(d, a0 + k, x[k]);
  }
}

// rest: only the units that k_md_advance does not take
__global__ void __launch_bounds__(256) k_md_units(const MdDesc *__restrict__ D, double dt, double hm, double h,
                                                  int flags, int rest) {
  const MdDesc &d = D[blockIdx.y];
  int u = blockIdx.x * blockDim.x + threadIdx.x;
  if (u >= (rest ? d.nrest : d.nunits)) return;
  if (rest) u = gmem(d.rest_unit)[u];
  flags = md_stage(d, flags);
  if (!(flags & ~MD_BETWEEN)) return;
  const int a0 = gmem(d.ufirst)[u];
  if (gmem(d.urigid)[u])
    md_unit<3>(d, u, a0, dt, hm, h, flags);
  else
    md_unit<1>(d, u, a0, dt, hm, h, flags);
}

// ---------------------------------------------------------------- a step's fast level in one launch

// A unit without terms: kicks, then nsub times drift, SHAKE, RATTLE (its fast forces are zero).
template <int NA>
__device__ __forceinline__ void md_free(const MdDesc &d, int a0, const double *dss, double dt, double hm, double h,
                                        int flags, int nsub) {
  double3 x[NA], v[NA];
  double m[NA], im[NA];
  md_load<NA>(d, a0, x, v, m, im);
  md_kicks<NA>(d, a0, dt, hm, flags, x, v, m, im);
  const double dti = h != 0.0 ? 1.0 / h : 0.0;
  for (int s = 0; s < nsub; ++s) {
    double3 p[NA];
#pragma unroll
    for (int k = 0; k < NA; ++k) {
      p[k] = x[k];
      x[k] = mim_fma(h, v[k], x[k]);
    }
    if constexpr (NA == 3) {
      if (!shake_mim3(x, p, im, dss, dti, v)) atomicAdd(d.fail, 1);
      rattle_mim3(x, v, im);
    }
  }
#pragma unroll
  for (int k = 0; k < NA; ++k) {
    md_store_v(d, a0 + k, v[k]);
    if (nsub) md_store_x(d, a0 + k, x[k]);
  }
}

// The atoms of one workgroup's slots (K a thread), connected by terms among
// themselves only: positions in LDS, everything else in registers.  An atom
// sums its own terms, in the order of the terms, from both ends' positions:
// twice the arithmetic of one thread per term, but no second pass.
template <int K>
__device__ __forceinline__ void md_connected(const MdDesc &d, int s0, int n, double (*pos)[3], double dt, double hm,
                                             double h, int flags, int nsub) {
  const double ts2 = h * h;
  double3 x[K][1], v[K][1], f[K];
  double m[K][1], im[K][1];
  int at[K], deg[K], off[K];
#pragma unroll
  for (int k = 0; k < K; ++k) {
    const int s = k * MD_WG + threadIdx.x;
    at[k] = s < n ? gmem(d.slot_atom)[s0 + s] : -1;
    deg[k] = off[k] = 0;
    if (at[k] < 0) continue;
    deg[k] = gmem(d.slot_deg)[s0 + s];
    off[k] = gmem(d.slice_off)[(s0 + s) >> 6] + (threadIdx.x & 63);
    md_load<1>(d, at[k], x[k], v[k], m[k], im[k]);
    f[k] = make_double3(gmem(d.bfx)[at[k]], gmem(d.bfy)[at[k]], gmem(d.bfz)[at[k]]);
    md_kicks<1>(d, at[k], dt, hm, flags, x[k], v[k], m[k], im[k]);
  }
  for (int s = 0; s < nsub; ++s) {
#pragma unroll
    for (int k = 0; k < K; ++k) {
      if (at[k] < 0) continue;
      double3 &xx = x[k][0], &vv = v[k][0];
      const double w = m[k][0];
      xx.x = xx.x + h * vv.x + f[k].x * 0.5 * ts2 / w;
      xx.y = xx.y + h * vv.y + f[k].y * 0.5 * ts2 / w;
      xx.z = xx.z + h * vv.z + f[k].z * 0.5 * ts2 / w;
      vv.x = vv.x + f[k].x * 0.5 * h / w;
      vv.y = vv.y + f[k].y * 0.5 * h / w;
      vv.z = vv.z + f[k].z * 0.5 * h / w;
      double *p = pos[k * MD_WG + threadIdx.x];
      p[0] = xx.x;
      p[1] = xx.y;
      p[2] = xx.z;
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < K; ++k) {
      if (at[k] < 0) continue;
      double3 &xx = x[k][0], &vv = v[k][0];
      double3 sum = make_double3(0.0, 0.0, 0.0);
#pragma unroll 2
      for (int e = 0; e < deg[k]; ++e) {
        const double *p = pos[gmem(d.ent_slot)[off[k] + 64 * e]];
        const double2 kr = gload(d.ent_kr + off[k] + 64 * e);
        const double dx = xx.x - p[0], dy = xx.y - p[1], dz = xx.z - p[2];
        const double r = sqrt(dx * dx + dy * dy + dz * dz);
        const double g = -2.0 * kr.x * (r - kr.y) / r;  // force along (x_i - x_j)
        {
#pragma clang fp contract(off)
          // each term's vector rounded before it is added, as k_md_bonds stores it
          sum.x = sum.x + g * dx;
          sum.y = sum.y + g * dy;
          sum.z = sum.z + g * dz;
        }
      }
      f[k] = sum;
      const double w = m[k][0];
      vv.x = vv.x + sum.x * 0.5 * h / w;
      vv.y = vv.y + sum.y * 0.5 * h / w;
      vv.z = vv.z + sum.z * 0.5 * h / w;
    }
    __syncthreads();
  }
#pragma unroll
  for (int k = 0; k < K; ++k) {
    if (at[k] < 0) continue;
    md_store_v(d, at[k], v[k][0]);
    if (!nsub) continue;
    md_store_x(d, at[k], x[k][0]);
    gmem(d.bfx)[at[k]] = f[k].x;
    gmem(d.bfy)[at[k]] = f[k].y;
    gmem(d.bfz)[at[k]] = f[k].z;
  }
}

// The kicks that end a step and start the next, then the next step's nsub fast
// substeps, in one launch; its workgroups take the connected atoms first, then
// MD_FREE units without terms each (a wavefront a SIMD: a unit's constraints
// are one serial chain of FP64 instructions, so spreading the units over the
// chip is what counts).  Four substeps of 216 waters: 11 us, where five
// launches over the units and four over the atoms took 42 and the gaps between
// them; of 4,900 waters and a 1,660-atom solute 19 us instead of 66.
__global__ void __launch_bounds__(MD_WG) k_md_advance(const MdDesc *__restrict__ D, int nconn, double dt, double hm,
                                                      double h, int flags, int nsub) {
  extern __shared__ __align__(16) double md_pos[];
  const MdDesc &d = D[blockIdx.y];
  const int blk = blockIdx.x;
  if (md_stage(d, flags) != flags) {
    flags = md_stage(d, flags);
    nsub = 0;
  }
  if (blk < nconn) {
    if (blk >= d.nwg) return;
    const int s0 = gmem(d.wg_slot)[blk], n = gmem(d.wg_slot)[blk + 1] - s0;
    double(*pos)[3] = reinterpret_cast<double(*)[3]>(md_pos);
    if (n <= MD_WG) md_connected<1>(d, s0, n, pos, dt, hm, h, flags, nsub);
    else md_connected<2>(d, s0, n, pos, dt, hm, h, flags, nsub);
    return;
  }
  const int u = (blk - nconn) * MD_FREE + threadIdx.x;
  if (threadIdx.x >= MD_FREE || u >= d.nfree) return;
  const int a0 = gmem(d.free_atom)[u];
  if (u < d.nfree_rigid) md_free<3>(d, a0, d.free_d2 + 3 * (size_t)u, dt, hm, h, flags, nsub);
  else md_free<1>(d, a0, nullptr, dt, hm, h, flags, nsub);
}

__global__ void __launch_bounds__(256) k_md_bonds(const MdDesc *__restrict__ D, int rest) {
  const MdDesc &d = D[blockIdx.y];
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= d.nbond || (rest && !d.nrest)) return;
  const int i = d.bi[t], j = d.bj[t];
  const double dx = d.x[i] - d.x[j], dy = d.y[i] - d.y[j], dz = d.z[i] - d.z[j];
  const double r = sqrt(dx * dx + dy * dy + dz * dz);
  const double dr = r - d.br0[t];
  const double f = -2.0 * d.bk[t] * dr / r;  // force on i along (x_i - x_j)
  d.bpf[3 * (size_t)t] = f * dx;
  d.bpf[3 * (size_t)t + 1] = f * dy;
  d.bpf[3 * (size_t)t + 2] = f * dz;
  d.bpe[t] = d.bk[t] * dr * dr;
}

// fast forces per atom from its terms, in fixed order
__global__ void __launch_bounds__(256) k_md_bond_gather(const MdDesc *__restrict__ D, int rest) {
  const MdDesc &d = D[blockIdx.y];
  const int a = blockIdx.x * blockDim.x + threadIdx.x;
  if (a >= d.natoms || (rest && !d.nrest)) return;
  double sx = 0.0, sy = 0.0, sz = 0.0;
  for (int t = d.bg_off[a]; t < d.bg_off[a + 1]; ++t) {
    const int sp = d.bg_term[t];
    const int p = (sp > 0 ? sp : -sp) - 1;
    const double s = sp > 0 ? 1.0 : -1.0;
    sx += s * d.bpf[3 * (size_t)p];
    sy += s * d.bpf[3 * (size_t)p + 1];
    sz += s * d.bpf[3 * (size_t)p + 2];
  }
  d.bfx[a] = sx;
  d.bfy[a] = sy;
  d.bfz[a] = sz;
}

// Per-system energies into d.out: [0] kinetic, [1] bond energy, [2..4]
// momentum; one block per component, fixed order over atoms / terms.
__global__ void __launch_bounds__(256) k_md_energy(const MdDesc *__restrict__ D) {
  __shared__ double red[4];
  const MdDesc &d = D[blockIdx.y];
  const int k = blockIdx.x;
  double s = 0.0;
  if (k == 1) {
    for (int t = threadIdx.x; t < d.nbond; t += blockDim.x) s += d.bpe[t];
  } else {
    for (int a = threadIdx.x; a < d.natoms; a += blockDim.x) {
      const double m = d.mass[a];
      if (k == 0) s += 0.5 * m * (d.vx[a] * d.vx[a] + d.vy[a] * d.vy[a] + d.vz[a] * d.vz[a]);
      else if (k == 2) s += m * d.vx[a];
      else if (k == 3) s += m * d.vy[a];
      else s += m * d.vz[a];
    }
  }
  s = wave_sum(s);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = s;
  __syncthreads();
  if (threadIdx.x == 0) {
    double t = 0.0;
    for (int w = 0; w < (int)(blockDim.x >> 6); ++w) t += red[w];
    d.out[k] = t;
  }
}

// steepest-descent relaxation step: each unit moves along its force by at
// most dmax (per atom h F/m capped at dmax), then SHAKE; velocities are zeroed
template <int NA>
__device__ __forceinline__ void md_relax_unit(const MdDesc &d, int u, int a0, double hstep, double dmax) {
  double3 x[NA], p[NA], dv[NA];
  double im[NA];
#pragma unroll
  for (int k = 0; k < NA; ++k) {
    const int a = a0 + k;
    im[k] = 1.0 / gmem(d.mass)[a];
    p[k] = make_double3(gmem(d.x)[a], gmem(d.y)[a], gmem(d.z)[a]);
    double fx = gmem(d.fx)[a] + gmem(d.bfx)[a], fy = gmem(d.fy)[a] + gmem(d.bfy)[a],
           fz = gmem(d.fz)[a] + gmem(d.bfz)[a];
    if (d.fmx) {
      fx += gmem(d.fmx)[a];
      fy += gmem(d.fmy)[a];
      fz += gmem(d.fmz)[a];
    }
    double sx = hstep * im[k] * fx, sy = hstep * im[k] * fy, sz = hstep * im[k] * fz;
    const double s = sqrt(sx * sx + sy * sy + sz * sz);
    if (!(s <= dmax)) {  // also catches a non-finite step
      const double c = s > 0.0 && s < 1e300 ? dmax / s : 0.0;
      sx *= c;
      sy *= c;
      sz *= c;
    }
    x[k] = make_double3(p[k].x + sx, p[k].y + sy, p[k].z + sz);
    dv[k] = make_double3(0.0, 0.0, 0.0);
  }
  if constexpr (NA == 3)
    if (!shake_mim3(x, p, im, d.ud2 + 3 * (size_t)u, 0.0, dv)) atomicAdd(d.fail, 1);
#pragma unroll
  for (int k = 0; k < NA; ++k) {
    const int a = a0 + k;
    gmem(d.x)[a] = x[k].x;
    gmem(d.y)[a] = x[k].y;
    gmem(d.z)[a] = x[k].z;
    gmem(d.vx)[a] = 0.0;
    gmem(d.vy)[a] = 0.0;
    gmem(d.vz)[a] = 0.0;
    double xp, yp, zp;
    to_reduced(d.oc, x[k].x, x[k].y, x[k].z, xp, yp, zp);
    gmem(d.xp)[a] = xp;
    gmem(d.yp)[a] = yp;
    gmem(d.zp)[a] = zp;
  }
}

// one steepest-descent step of every unit: displacement hstep F/m capped at
// dmax per atom, rigid units put back on their constraints, velocities zeroed
__global__ void __launch_bounds__(256) k_md_relax(const MdDesc *__restrict__ D, double hstep, double dmax) {
  const MdDesc &d = D[blockIdx.y];
  const int u = blockIdx.x * blockDim.x + threadIdx.x;
  if (u >= d.nunits) return;
  const int a0 = gmem(d.ufirst)[u];
  if (gmem(d.urigid)[u])
    md_relax_unit<3>(d, u, a0, hstep, dmax);
  else
    md_relax_unit<1>(d, u, a0, hstep, dmax);
}

// v *= scale (per system), e.g. for velocity rescaling during equilibration
__global__ void __launch_bounds__(256) k_md_scale_v(const MdDesc *__restrict__ D, const double *scale) {
  const MdDesc &d = D[blockIdx.y];
  const int a = blockIdx.x * blockDim.x + threadIdx.x;
  if (a >= d.natoms) return;
  const double s = scale[blockIdx.y];
  d.vx[a] *= s;
  d.vy[a] *= s;
  d.vz[a] *= s;
}

// the step count at which the run of nsteps that starts here ends
__global__ void k_md_begin(const MdDesc *__restrict__ D, int nsteps) {
  if (threadIdx.x == 0) D[blockIdx.y].step[1] = D[blockIdx.y].step[0] + nsteps;
}

static void md_dims(const MdDesc *h, int nsys, int &max_units, int &max_atoms, int &max_bonds) {
  max_units = max_atoms = max_bonds = 0;
  for (int s = 0; s < nsys; ++s) {
    max_units = std::max(max_units, h[s].nunits);
    max_atoms = std::max(max_atoms, h[s].natoms);
    max_bonds = std::max(max_bonds, h[s].nbond);
  }
}

void launch_md_units(const MdDesc *d, const MdDesc *h, int nsys, double dt, double hm, double hin, int flags,
                     hipStream_t st) {
  int mu, ma, mb;
  md_dims(h, nsys, mu, ma, mb);
  if (mu > 0) hipLaunchKernelGGL(k_md_units, dim3((mu + 255) / 256, nsys), dim3(256), 0, st, d, dt, hm, hin, flags, 0);
}

static void fast_forces(const MdDesc *d, const MdDesc *h, int nsys, bool rest, hipStream_t st) {
  int mu, ma, mb;
  md_dims(h, nsys, mu, ma, mb);
  if (mb > 0) hipLaunchKernelGGL(k_md_bonds, dim3((mb + 255) / 256, nsys), dim3(256), 0, st, d, rest ? 1 : 0);
  if (ma > 0) hipLaunchKernelGGL(k_md_bond_gather, dim3((ma + 255) / 256, nsys), dim3(256), 0, st, d, rest ? 1 : 0);
}

void launch_md_fast_forces(const MdDesc *d, const MdDesc *h, int nsys, hipStream_t st) {
  fast_forces(d, h, nsys, false, st);
}

void launch_md_begin(const MdDesc *d, int nsys, int nsteps, hipStream_t st) {
  hipLaunchKernelGGL(k_md_begin, dim3(1, nsys), dim3(64), 0, st, d, nsteps);
}

void launch_md_advance(const MdDesc *d, const MdDesc *h, int nsys, double dt, double hm, double hin, int flags,
                       int nsub, hipStream_t st) {
  int mw = 0, ms = 0, mf = 0, mr = 0;
  for (int s = 0; s < nsys; ++s) {
    mw = std::max(mw, h[s].nwg);
    ms = std::max(ms, h[s].wg_most);
    mf = std::max(mf, h[s].nfree);
    mr = std::max(mr, h[s].nrest);
  }
  const int nb = mw + (mf + MD_FREE - 1) / MD_FREE;
  if (nb > 0)
    hipLaunchKernelGGL(k_md_advance, dim3(nb, nsys), dim3(MD_WG), ms * 3 * sizeof(double), st, d, mw, dt, hm, hin,
                       flags, nsub);
  if (mr == 0) return;
  // units the launch above does not take: one launch per kick and substep
  const dim3 g((mr + 255) / 256, nsys), b(256);
  const int between = flags & MD_BETWEEN;
  hipLaunchKernelGGL(k_md_units, g, b, 0, st, d, dt, hm, hin, flags | (nsub > 0 ? MD_VERLET : 0), 1);
  for (int k = 0; k < nsub; ++k) {
    fast_forces(d, h, nsys, true, st);
    hipLaunchKernelGGL(k_md_units, g, b, 0, st, d, dt, hm, hin,
                       between | MD_KICK_FAST | (k + 1 < nsub ? MD_VERLET : 0), 1);
  }
}

void launch_md_energy(const MdDesc *d, int nsys, hipStream_t st) {
  hipLaunchKernelGGL(k_md_energy, dim3(5, nsys), dim3(256), 0, st, d);
}

void launch_md_relax(const MdDesc *d, const MdDesc *h, int nsys, double hstep, double dmax, hipStream_t st) {
  int mu, ma, mb;
  md_dims(h, nsys, mu, ma, mb);
  if (mu > 0) hipLaunchKernelGGL(k_md_relax, dim3((mu + 255) / 256, nsys), dim3(256), 0, st, d, hstep, dmax);
}

void launch_md_scale_v(const MdDesc *d, const MdDesc *h, int nsys, const double *scale, hipStream_t st) {
  int mu, ma, mb;
  md_dims(h, nsys, mu, ma, mb);
  if (ma > 0) hipLaunchKernelGGL(k_md_scale_v, dim3((ma + 255) / 256, nsys), dim3(256), 0, st, d, scale);
}

}  // namespace orac
