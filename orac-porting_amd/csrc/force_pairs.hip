// force_pairs.hip -- the direct-space pair kernel (force.f:235-870) on gfx950.
//
// One wavefront per owner group (k_pairs, below).  The neighbour list is full
// (both directions), so every atom's force is summed by its own wavefront: no
// atomics, and the order of every sum is fixed.
//
// Molecular virial.  force.f accumulates st += f_ab (x) (C_a - C_b - s) per pair
// (C = molecule centre, s = the group-pair image shift) and, for switched
// pairs, the S'V terms with C_a and -(C_b + s).  Summed over pairs this equals
//     sum_a F_a (x) C_a  -  sum_pairs f_ab (x) s  -  sum_switched x3 (x) s,
// with F_a the total direct force on atom a.  The kernel accumulates that
// form: the shift terms are nonzero only for pairs across the cell boundary,
// and the per-atom term is added once per atom after the force reduction.
#include <algorithm>
#include <cstdlib>
#include <string>
#include <type_traits>

#include "common.hpp"
#include "kernels.hpp"

namespace orac {

// A&S 7.1.26 (force.f:123-125)
#define AS_A1 0.2548296
#define AS_A2 -0.28449674
#define AS_A3 1.4214137
#define AS_A4 -1.453152
#define AS_A5 1.0614054
#define AS_QP 0.3275911

// The pair kernel's records in cell order (or, for coordinates that come with
// their centres, in group order): sorted position t holds group perm[t].
__global__ void __launch_bounds__(256) k_pack_sorted(const PairDesc *__restrict__ D) {
  const PairDesc &d = D[blockIdx.y];
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= d.ngrp) return;
  const int g = d.perm ? gmem(d.perm)[t] : t;
  const int f0 = gmem(d.gfirst)[g], n = gmem(d.glast)[g] - f0 + 1;
  const int sf = d.soff ? gmem(d.soff)[t] : f0;
  const double gx = gmem(d.xpg)[g], gy = gmem(d.ypg)[g], gz = gmem(d.zpg)[g];
  pack_head(d, t, g, sf, f0, n, gx, gy, gz);
  for (int k = 0; k < n; ++k) pack_atom(d, sf + k, f0 + k, gx, gy, gz);
}

template <typename P>
__device__ inline bool has_partner_in(P ex_off, P ex_idx, int a, int lo, int hi) {
  for (int t = ex_off[a]; t < ex_off[a + 1]; ++t) {
    int p = ex_idx[t];
    if (p >= lo && p <= hi) return true;
  }
  return false;
}

template <typename P>
__device__ inline bool is_excluded(P ex_off, P ex_idx, int a, int b) {
  for (int t = ex_off[a]; t < ex_off[a + 1]; ++t)
    if (ex_idx[t] == b) return true;
  return false;
}

// Pair arithmetic built on one reciprocal square root per pair.  FP64: the
// hardware reciprocal square root and reciprocal seeds refined by one
// Newton-Raphson step each (~1e-14 relative; the reference's 1/sqrt and
// divides are correctly rounded, and the difference stays far below the
// force tolerance) for a fraction of the instructions of an IEEE divide and
// square root, and the exponential by a polynomial (pair_exp2) in place of
// the libm routine.  FP32
// (mixed precision): the hardware reciprocal, reciprocal square root and
// exponential, 1-2 ulp each.  Pair distances are positive and finite, so no
// special cases arise.
template <typename T>
__device__ inline T pair_rsqrt(T x);
template <>
__device__ inline double pair_rsqrt<double>(double x) {
  const double r = __builtin_amdgcn_rsq(x);
  return fma(r, fma(-0.5 * x, r * r, 0.5), r);
}
template <>
__device__ inline float pair_rsqrt<float>(float x) { return __builtin_amdgcn_rsqf(x); }
template <typename T>
__device__ inline T pair_rcp(T x);
template <>
__device__ inline double pair_rcp<double>(double x) {
  const double q = __builtin_amdgcn_rcp(x);
  return fma(q, fma(-x, q, 1.0), q);
}
template <>
__device__ inline float pair_rcp<float>(float x) { return __builtin_amdgcn_rcpf(x); }
// a * b + c with c in a scalar register pair: the three-operand form, which
// leaves the polynomials' constants out of the vector registers (the compiler
// copies each constant to a fresh pair and accumulates into that)
__device__ __forceinline__ double fma_const(double a, double b, double c) {
  double d;
  asm("v_fma_f64 %0, %1, %2, %3" : "=v"(d) : "v"(a), "v"(b), "s"(c));
  return d;
}
// 2^y for the Ewald factor exp(-(alpha r)^2) = 2^(-alpha^2 log2(e) r^2), from
// the squared distance.  y = n + f, |f| <= 1/2 (exact), and 2^f = 1 + f q(f) with q of degree 8
// interpolating (2^f - 1) / f at the Chebyshev nodes (3.7e-14 relative).
template <typename T>
__device__ inline T pair_exp2(T y);
template <>
__device__ inline double pair_exp2<double>(double y) {
  const double n = __builtin_rint(y), f = y - n;
  double p = fma_const(f, 1.0203121047189341e-07, 1.3255224879317324e-06);
  p = fma_const(p, f, 1.525268684635191e-05);
  p = fma_const(p, f, 0.0001540345585244999);
  p = fma_const(p, f, 0.0013333558179042969);
  p = fma_const(p, f, 0.009618129159402565);
  p = fma_const(p, f, 0.055504108664760424);
  p = fma_const(p, f, 0.2402265069581299);
  p = fma_const(p, f, 0.6931471805599453);
  p = fma(p, f, 1.0);
  return __builtin_amdgcn_ldexp(p, (int)n);
}
template <>
__device__ inline float pair_exp2<float>(float y) { return __builtin_amdgcn_exp2f(y); }

// exp(-(alpha r)^2), r = rsq * rsqrt(rsq): FP64 from rsq, beside the reciprocal
// square root rather than after it.  FP32 from r: the seed's error (1 ulp) then
// enters with the opposite sign to that of the force's 1 / r^3, of which it takes
// part back; from rsq the Coulomb forces are 1 to 2 % further from 64 bits.
template <typename T>
__device__ __forceinline__ T pair_ewald_exp(const PairDesc &d, T rsq, T r) {
  if constexpr (sizeof(T) == 8) return pair_exp2<T>(T(d.ew_exp2) * rsq);
  else return pair_exp2<T>(T(d.ew_exp2) * (r * r));
}

// The A&S 7.1.26 polynomial of erfc at qt = 1 / (1 + p x), without its exponential
template <typename T>
__device__ __forceinline__ T erfc_poly(T qt) {
  if constexpr (sizeof(T) == 8) {
    double p = fma_const(qt, AS_A5, AS_A4);
    p = fma_const(p, qt, AS_A3);
    p = fma_const(p, qt, AS_A2);
    p = fma_const(p, qt, AS_A1);
    return p * qt;
  } else {
    return ((((T(AS_A5) * qt + T(AS_A4)) * qt + T(AS_A3)) * qt + T(AS_A2)) * qt + T(AS_A1)) * qt;
  }
}

// force.f:486-490: two atoms at or above massinfty are skipped only where the
// list owner's atom has an exclusion partner in the other group (the owner is
// the lower group).  a: the owner atom (flags fa) of the group at sorted
// position t, atoms ia0 .. ia0 + nI - 1; ib: the neighbour atom's record.
__device__ __noinline__ bool heavy_masked(const PairDesc &d, int a, int fa, int t, int ia0, int nI, int2 ib, int tj) {
  const int b = ib.y;
  if (gmem(d.mass)[b] < d.massinfty || gmem(d.mass)[a] < d.massinfty) return false;
  const int g = d.perm ? gmem(d.perm)[t] : t, j = d.perm ? gmem(d.perm)[tj] : tj;
  if (j > g)
    return (fa & ATOM_EX) && has_partner_in(gmem(d.ex_off), gmem(d.ex_idx), a, gmem(d.gfirst)[j], gmem(d.glast)[j]);
  return (ib.x & ATOM_EX) && has_partner_in(gmem(d.ex_off), gmem(d.ex_idx), b, ia0, ia0 + nI - 1);
}

// Group-pair geometry (force.f:265-292): the image shift s (even integers in
// reduced units) and the centre separation after it, without contraction.
struct GroupGeom {
  double sxm, sym, szm, xcc, ycc, zcc, drj;
};
__device__ __forceinline__ GroupGeom group_geom(double xpgi, double ypgi, double zpgi, const double4 &gpj,
                                                const double *co) {
#pragma clang fp contract(off)
  GroupGeom g;
  double xgg = xpgi - gpj.x, ygg = ypgi - gpj.y, zgg = zpgi - gpj.z;
  g.sxm = g.sym = g.szm = 0.0;
  // dnint(d / 2) is zero below |d| = 1: a wavefront without a larger
  // difference (an owner away from the cell's faces) skips the rounding
  if (__ballot(!(fmax(fmax(fabs(xgg), fabs(ygg)), fabs(zgg)) < 1.0))) {
    g.sxm = 2.0 * fnint(0.5 * xgg);
    g.sym = 2.0 * fnint(0.5 * ygg);
    g.szm = 2.0 * fnint(0.5 * zgg);
    xgg = xgg - g.sxm;
    ygg = ygg - g.sym;
    zgg = zgg - g.szm;
  }
  g.xcc = co[0] * xgg + co[3] * ygg + co[6] * zgg;
  g.ycc = co[4] * ygg + co[7] * zgg;
  g.zcc = co[8] * zgg;
  g.drj = g.xcc * g.xcc + g.ycc * g.ycc + g.zcc * g.zcc;
  return g;
}

// The group pair is inside the shell: normal [rinn0, rout) or switched
// [rout, rout0) and [rinn, rinn0) (force.f:293-335), one interval since
// rinn <= rinn0 < rout <= rout0 (force.f:166 computes nothing otherwise).
__device__ __forceinline__ bool in_shell(const PairDesc &d, double drj) { return drj >= d.r2inn && drj < d.r2out0; }

// LJ {c12, c6} of the type pair (ti, tj), zero when c6 <= 1e-12 (the pair then
// has no LJ term, force.f:455; the dense tables hold such entries as zeros)
template <typename T, bool DENSE = false>
__device__ __forceinline__ void pair_lj(const PairDesc &d, int ti, int tj, T &c12, T &c6) {
  if (sizeof(T) == 4 && (DENSE || d.lj_dense32)) {
    const float2 v = gload_at(d.lj_dense32 + (size_t)ti * d.ntypes, tj);
    c12 = T(v.x);
    c6 = T(v.y);
  } else if (DENSE || d.lj_dense) {
    const double2 v = gload_at(d.lj_dense + (size_t)ti * d.ntypes, tj);
    c12 = T(v.x);
    c6 = T(v.y);
  } else {
    const int lij = gmem(d.type_table)[ti + (size_t)d.ntypes * tj];
    const double a = gmem(d.ecc12)[lij], b = gmem(d.ecc6)[lij];
    const bool lj = b > 1e-12;
    c12 = lj ? T(a) : T(0);
    c6 = lj ? T(b) : T(0);
  }
}

// One atom pair in soft-core form (force_alchemy.f:439-523): F = the pair's
// row of alch_fac, ap = {1 / sigma^6, epsmin, typeaij + 4} of its classes.
// LJ eps (gp^-2 - gp^-1) with gp = ljsoft f1 + r^6 / sigma^6, scaled by f2;
// Coulomb q_a q_b fq2 erfc(alpha r) / sqrt(qsoft fq1^2 + r^2) (or without
// erfc, plain); the energies at lambda0 come from the same distances with
// the lambda0 factors.  dw = U(lambda) - U(lambda0) of the pair.
template <typename T>
struct AlchTerms {
  T qf, conf, cou;
  double dw;
};

template <typename T>
__device__ __forceinline__ AlchTerms<T> alch_terms(const PairDesc &d, T xc, T yc, T zc, T qq, const double4 &ap,
                                                   const double *F) {
  const T rsq = xc * xc + yc * yc + zc * zc;
  const T rinv = pair_rsqrt<T>(rsq);
  T qforce = T(0), conf = T(0), conf0 = T(0), cou = T(0), cou0 = T(0);
  if (d.alch_shifted) {
    // force_alchemy_shifted.f:469-509: LJ at r + ljshift 2^(1/6) sigma f1, Coulomb over
    // r + qshift fq1 (erfc of the real distance)
    const T r = rsq * rinv;
    if (ap.y > 1e-12) {
      const T sig = T(ap.w), eps = T(ap.y);
      const T irl = pair_rcp<T>(r + T(F[0]) * sig), irl0 = pair_rcp<T>(r + T(F[2]) * sig);
      const T x = sig * irl, x2 = x * x, r6 = x2 * x2 * x2;
      const T y = sig * irl0, y2 = y * y, r60 = y2 * y2 * y2;
      qforce = T(F[1]) * eps * (T(12) * r6 * r6 - T(6) * r6) * (rinv * irl);
      conf = T(F[1]) * (eps * (r6 * r6 - r6));
      conf0 = T(F[3]) * (eps * (r60 * r60 - r60));
    }
    const T irq = pair_rcp<T>(r + T(F[4])), irq0 = pair_rcp<T>(r + T(F[6]));
    if (!d.lskip_ewald) {
      const T alphar = T(d.alpha) * r;
      const T qt = pair_rcp<T>(T(1) + T(AS_QP) * alphar);
      const T expcst = pair_ewald_exp<T>(d, rsq, r);
      const T erfcst = ((((T(AS_A5) * qt + T(AS_A4)) * qt + T(AS_A3)) * qt + T(AS_A2)) * qt + T(AS_A1)) * qt * expcst;
      const T furpar = T(F[5]) * qq;
      cou = furpar * erfcst * irq;
      cou0 = T(F[7]) * qq * erfcst * irq0;
      qforce += furpar * (rinv * irq) * (erfcst * irq + T(d.twrtpi) * alphar * expcst * rinv);
    } else if (!d.ewald) {
      cou = T(F[5]) * qq * irq;
      cou0 = T(F[7]) * qq * irq0;
      qforce += cou * (irq * rinv);
    }
  } else {
    const T auxaa = pair_rsqrt<T>(T(F[4]) + rsq);
    const T auxa0 = pair_rsqrt<T>(T(F[6]) + rsq);
    if (ap.y > 1e-12) {
      const T r6 = rsq * rsq * rsq * T(ap.x);
      const T gp1 = pair_rcp<T>(T(F[0]) + r6), gp2 = gp1 * gp1;
      const T gp10 = pair_rcp<T>(T(F[2]) + r6), gp20 = gp10 * gp10;
      const T eps = T(ap.y);
      const T ssvir = T(F[1]) * eps * (T(2) * gp1 * gp2 - gp2);
      qforce = T(6) * r6 * ssvir * (rinv * rinv);
      conf = T(F[1]) * (eps * (gp2 - gp1));
      conf0 = T(F[3]) * (eps * (gp20 - gp10));
    }
    if (!d.lskip_ewald) {
      const T r = rsq * rinv, alphar = T(d.alpha) * r;
      const T qt = pair_rcp<T>(T(1) + T(AS_QP) * alphar);
      const T expcst = pair_ewald_exp<T>(d, rsq, r);
      const T erfcst = ((((T(AS_A5) * qt + T(AS_A4)) * qt + T(AS_A3)) * qt + T(AS_A2)) * qt + T(AS_A1)) * qt * expcst;
      const T furpar = T(F[5]) * qq, furpar0 = T(F[7]) * qq;
      cou = furpar * erfcst * auxaa;
      cou0 = furpar0 * erfcst * auxa0;
      qforce += furpar * auxaa * (erfcst * (auxaa * auxaa) + T(d.twrtpi) * alphar * expcst * (rinv * rinv));
    } else if (!d.ewald) {
      cou = T(F[5]) * qq * auxaa;
      cou0 = T(F[7]) * qq * auxa0;
      qforce += cou * (auxaa * auxaa);
    }
  }
  AlchTerms<T> r;
  r.qf = qforce;
  r.conf = conf;
  r.cou = cou;
  r.dw = (double)(conf - conf0) + (double)(cou - cou0);
  return r;
}

// One plain atom pair: the force over the separation (force = qf * (x, y, z))
// and the two energies.  Every fused operation is written out, here and in the
// sums, so that all forms of the kernel round alike: a system's results do not
// depend on the systems beside it.
template <typename T>
struct PairTerms {
  T qf, conf, cou;
};

template <typename T>
__device__ __forceinline__ PairTerms<T> plain_terms(const PairDesc &d, T x, T y, T z, T qq, bool lskip, bool plainq,
                                                    bool lj, T c12, T c6) {
#pragma clang fp contract(off)
  const T rsq = fma(z, z, fma(y, y, x * x));
  const T rinv = pair_rsqrt<T>(rsq);
  const T rsqi = rinv * rinv;
  PairTerms<T> p;
  p.conf = T(0);
  if (!lskip) {
    const T r = rsq * rinv, expcst = pair_ewald_exp<T>(d, rsq, r);
    const T erfcst = erfc_poly<T>(pair_rcp<T>(fma(T(d.ew_qp), r, T(1)))) * expcst;
    const T qr = qq * rinv;
    p.cou = qr * erfcst;
    p.qf = fma(T(d.ew_twa) * r, expcst, erfcst) * (qr * rsqi);
  } else {
    p.cou = plainq ? qq * rinv : T(0);
    p.qf = p.cou * rsqi;
  }
  if (lj) {
    // FP32: from rsq, whose power rounds without the seed's bias (12 to 14 times it in rinv's
    // powers, which showed in the energy and the stress)
    const T r6 = sizeof(T) == 4 ? pair_rcp<T>(rsq * rsq * rsq) : rsqi * rsqi * rsqi;
    const T e6 = c6 * r6, e12 = c12 * r6 * r6;
    p.conf = e12 - e6;
    p.qf = fma(fma(T(12), e12, T(-6) * e6), rsqi, p.qf);
  }
  return p;
}

constexpr int PAIR_NACC = 16;      // energies and virial of a block: uconf[3], ucoul[3], st[9], dwrk

// ================================================================ k_pairs
//
// The lanes of a wavefront take the atoms of the owner's in-shell neighbour
// groups, one atom each, and loop over the owner group's atoms, whose records
// are the same across the wavefront and sit in LDS: a pair costs a few
// additions before its distance and reads no memory but its LJ entry, and a
// neighbour atom's record is read once for all owner atoms.  The list entries
// are classified 64 at a time; a kept entry's Cartesian group separation,
// image shift and switch are computed once and kept in a small LDS ring, and
// its atoms are appended to a ring of lane slots, from which passes of 64 are
// taken, so that every lane of a pass has an atom (the last pass aside),
// whatever the sizes of the groups.
//
// Bound by VALU issue (about 60 FP64 instructions and two quarter-rate seeds
// per pair, no matrix instruction fits a scalar function of each distance).
// What keeps the count down:
//  * an owner atom whose LJ row is empty (water hydrogens) skips the LJ gather
//    and arithmetic, a wave-uniform branch;
//  * the S'(r) V term of switched group pairs is linear in V, so each lane
//    adds its own share -S'(r)/r v (C_i - C_j) and no lane needs the group
//    pair's total;
//  * the list is full, so every pair is seen from both sides: energies and
//    image-shift virial are summed over both and halved, with no test which
//    side counts;
//  * exclusions of an owner atom are walked as a wave-uniform loop;
//  * the 64-lane sums go through LDS eight values at a time (8 writes, 8 reads
//    per lane and three exchanges for eight sums).
// Measured on the 24,460-atom system (11.9 M pair evaluations from both sides):
// 85 us in FP64 and 78 us in FP32, against 182 and 155 us with lanes on (owner
// atom, neighbour group) that recomputed the group geometry per lane; 27 M
// vector instructions (26 M in FP32) against 43 M.  16 systems in one launch:
// 58 us each (FP32).  FP32 separations from a rounded centre separation that
// differed between a pair's two sides took 2.5% less at 103,000 atoms (236 us,
// now 242), but the two forces of a pair did not cancel, and what they left
// made the virial's error 1.6e-7 for 0.5e-7 (24,460 atoms; 2.4 for 1.2 at 103,000).

constexpr int ENT_RING = 128;   // entries kept: at most 63 with atoms waiting + 64 new ones
constexpr int SLOT_RING = 256;  // lane slots: at most 63 waiting + one round's atoms
constexpr int RED_STRIDE = 72;  // 8 rows of 64 values, rows 16 banks apart

// U: owner atoms whose sums stay in registers during a list walk
template <int U>
struct PairWave {
  double gx[ENT_RING], gy[ENT_RING], gz[ENT_RING];  // centre separation, image applied (R = float: {hi, lo} floats)
  double sw[ENT_RING], dsw[ENT_RING];               // S and S'(r) / r of the group distance (1 and 0 unswitched)
  int sx[ENT_RING], sy[ENT_RING], sz[ENT_RING];     // image shift (even integers, reduced units)
  int bs[ENT_RING];                                 // sorted first atom | solute neighbour << 26 | shifted << 27
  int tj[ENT_RING];                                 // neighbour group, sorted position
  unsigned short slot[SLOT_RING];                   // entry | atom within the group << 7
  double4 own[U];                                   // the owner atoms' records (R = float: four floats)
};
static_assert(sizeof(PairWave<1>) >= 8 * RED_STRIDE * sizeof(double), "the lane sums reuse the ring");

template <int U>
struct PairShared {
  PairWave<U> w[PAIR_WAVES];
  double fsum[PAIR_WAVES][64][3];          // owner-atom forces of a wave's part of the list
  double red[PAIR_WAVES][3 + PAIR_NACC];   // S'V vector, then energies and virial
  double alch[9][8];                       // the system's soft-core factors (alchemical kernels)
};

// A wave-uniform value the compiler must take anew here: tests of it stay at
// their place instead of being held in (and spilled from) scalar registers
// across the whole list walk.
__device__ __forceinline__ int here(int v) {
  asm volatile("" : "+s"(v));
  return v;
}

// Sums of eight values over the 64 lanes; lane l returns the sum of v[l >> 3].
// Fixed order: lane l adds the eight lanes = l mod 8, then lanes 1, 2, 4 apart.
__device__ __forceinline__ double wave_sum8(const double *v, double *buf, int lane) {
  wave_lds_sync();
#pragma unroll
  for (int k = 0; k < 8; ++k) buf[k * RED_STRIDE + lane] = v[k];
  wave_lds_sync();
  const double *row = buf + (lane >> 3) * RED_STRIDE + (lane & 7);
  double s = row[0];
#pragma unroll
  for (int k = 1; k < 8; ++k) s += row[8 * k];
  s += __shfl_xor(s, 1, 64);
  s += __shfl_xor(s, 2, 64);
  s += __shfl_xor(s, 4, 64);
  return s;
}

// An atom's Cartesian offset from its group centre and its charge, in the pair precision.
template <typename T>
struct AtomRec {
  T x, y, z, q;
};
template <typename T>
__device__ __forceinline__ AtomRec<T> atom_rec(const PairDesc &d, int s) {
  if constexpr (sizeof(T) == 4) {
    const float4 v = gload_at(d.sapf, s);
    return {v.x, v.y, v.z, v.w};
  } else {
    const double4 v = gload_at(d.sapc, s);
    return {v.x, v.y, v.z, v.w};
  }
}

// The pair forms of a kernel: plain (every system with the Ewald term, a dense
// LJ table and no atom at massinfty: what a simulation runs), soft core
// (alchemical systems), REM segment scaling, and plain without those limits
// (an outer shell that skips the Ewald term, more than LJ_DENSE_MAX types).
enum { PAIR_PLAIN = 0, PAIR_ALCH = 1, PAIR_REM = 2, PAIR_ANY = 3 };

// Owner atoms a list walk takes (their sums stay in registers).  Three suit
// waters and charge groups of a few atoms; groups of dozens of atoms walk their
// list again for every three and have so few owners that eight at half the
// occupancy are better.  13,824 to 21,952 atoms, us with 3 and with 8 (FP64;
// FP32), and before the lanes took the neighbours: groups of 6 atoms 64 71 (88);
// 54 62 (58), of 8 80 80 (80); 68 68 (64), of 12 115 92 (107); 103 80 (90), of 16
// 178 121 (148); 161 102 (123), of 64 1,530 900 (1,046); 1,458 836 (919).
constexpr int OWN_FEW = 3, OWN_MANY = 8;
int pair_many_for(int natoms, int ngrp) { return (long long)natoms > 8ll * ngrp ? 1 : 0; }

// One work item: block blk of system d (PAIR_WAVES waves, split of them per owner group).
template <typename T, int MODE, int U>
__device__ __forceinline__ void pairs_item(const PairDesc &d, int blk, PairShared<U> &sh) {
  if (blk >= d.nblk || d.half || (d.many != 0) != (U == OWN_MANY)) return;
  // Separations and charge products: alchemical systems form them in FP64 and round once, also where
  // the pair arithmetic is FP32 (a window's dU/dlambda is a small difference of large terms).
  using R = std::conditional_t<MODE == PAIR_ALCH, double, T>;
  constexpr bool F32 = sizeof(R) == 4;
  constexpr bool DW = MODE == PAIR_ALCH || MODE == PAIR_REM;  // a 16th sum: dwrk or the segment energy
  if (MODE == PAIR_ALCH) {
    if (threadIdx.x < 72) sh.alch[threadIdx.x >> 3][threadIdx.x & 7] = gmem(d.alch_fac)[threadIdx.x];
    __syncthreads();
  }
  // (wave-uniform for the compiler too: the loop control then stays in scalar registers)
  const int lane = threadIdx.x & 63, wid = uniform((int)(threadIdx.x >> 6));
  // S waves share one owner group, each taking a contiguous part of its list
  const int S = d.split, part = wid % S;
  const int t = uniform(blk * (PAIR_WAVES / S) + wid / S);  // owner group, sorted position
  PairWave<U> &W = sh.w[wid];
  double *buf = reinterpret_cast<double *>(&W);
  double x3[3] = {0.0, 0.0, 0.0};                 // S'(r) V vectors of the switched group pairs
  double ec[2] = {0.0, 0.0}, eq[2] = {0.0, 0.0};  // LJ and Coulomb energy by the neighbour's class
  double st[9], dwl = 0.0;
#pragma unroll
  for (int k = 0; k < 9; ++k) st[k] = 0.0;
  bool any_st = false;                            // wave-uniform
  int ia0 = 0, nI = 0, typei = 1;
  if (t < d.ngrp) {
    const double4 gpi = gload(d.sgp + t);
    const double xpgi = uniform(gpi.x), ypgi = uniform(gpi.y), zpgi = uniform(gpi.z);
    int gw[2];
    __builtin_memcpy(gw, &gpi.w, 8);
    const int as0 = uniform(gw[0]);
    nI = uniform(gw[1] & 255);
    typei = uniform(gw[1] >> 8);
    ia0 = uniform(gload_at(d.sai, as0).y);
    int nb0, nb1;
    if (d.nb_slab > 0) {
      nb0 = t * d.nb_slab;
      nb1 = nb0 + min(uniform(gmem(d.nb_cnt)[t]), d.nb_slab);
    } else {
      nb0 = uniform(gmem(d.nb_off)[t]);
      nb1 = uniform(gmem(d.nb_off)[t + 1]);
    }
    if (S > 1) {
      const int len = nb1 - nb0;
      nb1 = nb0 + (len * (part + 1)) / S;
      nb0 = nb0 + (len * part) / S;
    }
    // entries per classification round: all of a round's atoms fit the slots beside 63 waiting ones
    const int mg = d.max_group;
    const int per_round = min(64, (SLOT_RING - 63) / mg);
    const bool lskip = (MODE == PAIR_ALCH || MODE == PAIR_ANY) && d.lskip_ewald != 0, plainq = !d.ewald;
    const double inv_o2 = d.inv_arsout2, inv_i2 = d.inv_arsinn2;
    for (int u0 = 0; u0 < nI; u0 += U) {
      const int nu = min(U, nI - u0);
      int ot[U];  // type << ATOM_FLAG_BITS | flags
      int xn[U], xv[U];
      double fr[U][3];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int a = as0 + u0 + min(u, nu - 1);
        const AtomRec<R> r = atom_rec<R>(d, a);
        if (lane == 0) __builtin_memcpy(&W.own[u], &r, sizeof r);
        ot[u] = uniform(gload_at(d.sai, a).x);
        fr[u][0] = fr[u][1] = fr[u][2] = 0.0;
        // an atom with exclusions outside its group: the first 64, one a lane
        xn[u] = 0;
        xv[u] = -1;
        if (ot[u] & ATOM_EX) {
          const int x0 = uniform(gmem(d.ex_off)[ia0 + u0 + min(u, nu - 1)]);
          xn[u] = uniform(gmem(d.ex_off)[ia0 + u0 + min(u, nu - 1) + 1]) - x0;
          if (lane < xn[u]) xv[u] = gmem(d.ex_idx)[x0 + lane];
        }
      }
      int c0 = nb0, ecount = 0, shead = 0, ns = 0;
      for (;;) {
        while (ns < 64 && c0 < nb1) {
          // ---- classify per_round entries; the in-shell ones are kept in list order
          const int jj = c0 + lane;
          const bool in = lane < per_round && jj < nb1;
          c0 += per_round;
          const int tj = in ? gmem(d.nb_idx)[jj] : t;
          const double4 gpj = gload_at(d.sgp, tj);
          const GroupGeom gg = group_geom(xpgi, ypgi, zpgi, gpj, d.co);
          const bool keep = in && in_shell(d, gg.drj);
          int jw[2];
          __builtin_memcpy(jw, &gpj.w, 8);
          const int nJ = keep ? (jw[1] & 255) : 0;
          const unsigned long long m = __ballot(keep);
          // exclusive prefix of the kept entries' atom counts, one bit of the counts at a time
          int apos = 0, atot = 0;
          for (int b = 0; (mg >> b) != 0; ++b) {
            const unsigned long long mb = __ballot((nJ >> b) & 1);
            apos += lanes_below(mb) << b;
            atot += __popcll(mb) << b;
          }
          if (keep) {
            const int e = (ecount + lanes_below(m)) & (ENT_RING - 1);
            double sw = 1.0, dsw = 0.0;
            if (!(gg.drj >= d.r2inn0 && gg.drj < d.r2out)) {
              const double rinv = pair_rsqrt<double>(gg.drj), rsp = gg.drj * rinv;
              if (gg.drj >= d.r2out && gg.drj < d.r2out0) {
                const double auxa = (d.arsout1 + 2.0 * rsp) * inv_o2, auxb = d.rout0 - rsp;
                sw = auxa * (auxb * auxb);
                dsw = fma(2.0 * (auxb * auxb), inv_o2, -(2.0 * auxa * auxb)) * rinv;
              } else {
                const double auxa = (d.arsinn1 + 2.0 * rsp) * inv_i2, auxb = d.rinn0 - rsp;
                sw = fma(-auxa, auxb * auxb, 1.0);
                dsw = -fma(2.0 * (auxb * auxb), inv_i2, -(2.0 * auxa * auxb)) * rinv;
              }
            }
            if constexpr (F32) {
              float2 g;
              g.x = (float)gg.xcc;
              g.y = (float)(gg.xcc - (double)g.x);
              __builtin_memcpy(&W.gx[e], &g, 8);
              g.x = (float)gg.ycc;
              g.y = (float)(gg.ycc - (double)g.x);
              __builtin_memcpy(&W.gy[e], &g, 8);
              g.x = (float)gg.zcc;
              g.y = (float)(gg.zcc - (double)g.x);
              __builtin_memcpy(&W.gz[e], &g, 8);
            } else {
              W.gx[e] = gg.xcc;
              W.gy[e] = gg.ycc;
              W.gz[e] = gg.zcc;
            }
            W.sw[e] = sw;
            W.dsw[e] = dsw;
            const bool shifted = gg.sxm != 0.0 || gg.sym != 0.0 || gg.szm != 0.0;
            if (shifted) {
              W.sx[e] = (int)gg.sxm;
              W.sy[e] = (int)gg.sym;
              W.sz[e] = (int)gg.szm;
            }
            W.bs[e] = jw[0] | ((jw[1] >> 8) == 1 ? 1 << 26 : 0) | (shifted ? 1 << 27 : 0);
            if (MODE != PAIR_PLAIN) W.tj[e] = tj;
            const int s0 = shead + ns + apos;
            for (int k = 0; k < mg; ++k)
              if (k < nJ) W.slot[(s0 + k) & (SLOT_RING - 1)] = (unsigned short)(e | (k << 7));
          }
          ecount += __popcll(m);
          ns += atot;
        }
        if (ns <= 0) break;
        wave_lds_sync();
        // ---- one pass: up to 64 neighbour atoms
        const int np = min(ns, 64);
        const bool have = lane < np;
        const int sl = W.slot[(shead + (have ? lane : 0)) & (SLOT_RING - 1)];
        const int e = sl & 127, k = sl >> 7;
        const int eb = W.bs[e];
        const int js = (eb & 0x3ffffff) + k;
        const AtomRec<R> rb = atom_rec<R>(d, js);
        const int2 ib = gload_at(d.sai, js);
        const double sw = have ? W.sw[e] : 0.0, dsw = have ? W.dsw[e] : 0.0;
        // separation = owner centre - neighbour centre - image (bx) + owner offset - neighbour offset.  FP32
        // pairs: the centre separation as hi + lo (or FP64), and every rounding the same from either
        // side, so that a pair's two forces cancel exactly and leave no net force to the virial
        R bx, by, bz, lx, ly, lz;
        if constexpr (F32) {
          float2 g;
          __builtin_memcpy(&g, &W.gx[e], 8);
          bx = g.x;
          lx = g.y;
          __builtin_memcpy(&g, &W.gy[e], 8);
          by = g.x;
          ly = g.y;
          __builtin_memcpy(&g, &W.gz[e], 8);
          bz = g.x;
          lz = g.y;
        } else {
          bx = W.gx[e];
          by = W.gy[e];
          bz = W.gz[e];
          if constexpr (sizeof(T) == 8) {
            bx -= rb.x;
            by -= rb.y;
            bz -= rb.z;
          }
        }
        const bool shifted = have && ((eb >> 27) & 1) != 0, solute = ((eb >> 26) & 1) != 0;
        const bool pass_st = __ballot(shifted) != 0ull, pass_solute = __ballot(have && solute) != 0ull;
        const bool pass_ex = __ballot((ib.x & ATOM_EX) != 0) != 0ull;
        any_st = any_st || pass_st;
        const int tb = ib.x >> ATOM_FLAG_BITS;
        // the first owner atom's LJ entry (a water's only one), requested before the arithmetic that hides it
        T c12a = T(0), c6a = T(0);
        if (ot[0] & ATOM_LJ) pair_lj<T, MODE == PAIR_PLAIN>(d, ot[0] >> ATOM_FLAG_BITS, tb, c12a, c6a);
        double vc = 0.0, vq = 0.0, fsx = 0.0, fsy = 0.0, fsz = 0.0, seg = 0.0, vr = 0.0;
        auto owner_atoms = [&](auto st_tag) {
          constexpr bool ST = decltype(st_tag)::value;
#pragma unroll
          for (int u = 0; u < U; ++u) {
            if (u < nu) {
              const int fl = here(ot[u]);
              AtomRec<R> ra;
              __builtin_memcpy(&ra, &W.own[u], sizeof ra);
              T x, y, z;
              if constexpr (sizeof(T) == 8) {
                x = bx + ra.x;
                y = by + ra.y;
                z = bz + ra.z;
              } else if constexpr (F32) {
                x = bx + (lx + (ra.x - rb.x));
                y = by + (ly + (ra.y - rb.y));
                z = bz + (lz + (ra.z - rb.z));
              } else {
                x = T(bx + (ra.x - rb.x));
                y = T(by + (ra.y - rb.y));
                z = T(bz + (ra.z - rb.z));
              }
              T qq = T(ra.q * rb.q);
              bool masked = false;
              const bool heavy = MODE != PAIR_PLAIN && d.any_heavy != 0;
              if (((fl & ATOM_EX) && pass_ex) || heavy) {  // wave-uniform
                const int a = ia0 + u0 + u;
                if ((fl & ATOM_EX) && pass_ex) {  // the owner atom's exclusions
                  const int nx = min(xn[u], 64);
                  for (int q = 0; q < nx; ++q) masked |= __builtin_amdgcn_readlane(xv[u], q) == ib.y;
                  for (int q = 64; q < xn[u]; ++q) masked |= gmem(d.ex_idx)[gmem(d.ex_off)[a] + q] == ib.y;
                }
                if (heavy) masked |= heavy_masked(d, a, fl, t, ia0, nI, ib, W.tj[e]);
                // no charge, no LJ, and a distance that keeps the zeros finite
                qq = masked ? T(0) : qq;
                x = masked ? T(1) : x;
              }
              T qf, cou, conf;
              double dw = 0.0;
              // (per lane: a pair takes the same form from either side)
              if (MODE == PAIR_ALCH && ((fl | ib.x) & ATOM_ALCH)) {
                const double4 ap = gload_at(d.alch_pair, (fl >> ATOM_FLAG_BITS) * d.ntypes + tb);
                const AlchTerms<T> r = alch_terms<T>(d, x, y, z, qq, ap, sh.alch[(int)ap.z]);
                // (the soft core takes its own parameters)
                qf = masked ? T(0) : r.qf;
                conf = masked ? T(0) : r.conf;
                cou = masked ? T(0) : r.cou;
                dw = masked ? 0.0 : r.dw;
              } else {
                const bool lj = (fl & ATOM_LJ) != 0;  // some type has LJ with this owner atom's
                T c12 = c12a, c6 = c6a;
                if (lj) {
                  if (u > 0) pair_lj<T, MODE == PAIR_PLAIN>(d, fl >> ATOM_FLAG_BITS, tb, c12, c6);
                  c12 = masked ? T(0) : c12;
                  c6 = masked ? T(0) : c6;
                }
                const PairTerms<T> r = plain_terms<T>(d, x, y, z, qq, lskip, plainq, lj, c12, c6);
                qf = r.qf;
                conf = r.conf;
                cou = r.cou;
              }
              if (MODE == PAIR_ALCH) seg += dw;
              if (MODE == PAIR_ALCH || (fl & ATOM_LJ)) vc += (double)conf;
              vq += (double)cou;
              double w = (double)qf * sw;
              if (MODE == PAIR_REM) {
                // force_REM.f:491-494, 649-664, 679-682 (Ewald branch): a selected pair's force is scaled by
                // rem_f3 and its energy goes to the segment energy; its share of V for the switch derivative
                // is scaled too (cmap2), the shell energies are not
                const bool ra = (fl & ATOM_REM) != 0, rbs = (ib.x & ATOM_REM) != 0;
                const bool sel = d.rem_kind == 0 ? (ra || rbs) : (d.rem_kind == 1 ? (ra && rbs) : (ra != rbs));
                const double f = sel ? d.rem_f3 : 1.0, en = (double)conf + (double)cou;
                w *= f;
                if (sel) seg += en;
                vr += f * en;
              }
              fr[u][0] = fma(w, (double)x, fr[u][0]);
              fr[u][1] = fma(w, (double)y, fr[u][1]);
              fr[u][2] = fma(w, (double)z, fr[u][2]);
              if (ST) {
                fsx = fma(w, (double)x, fsx);
                fsy = fma(w, (double)y, fsy);
                fsz = fma(w, (double)z, fsz);
              }
            }
          }
        };
        // the image-shift virial needs the lane's summed force: a path of its own
        if (pass_st)
          owner_atoms(std::true_type{});
        else
          owner_atoms(std::false_type{});
        // ---- the lane's share of the group pair's energies, S'V term and image-shift virial
        if (pass_solute) {
          ec[0] += solute ? sw * vc : 0.0;
          eq[0] += solute ? sw * vq : 0.0;
          ec[1] += solute ? 0.0 : sw * vc;
          eq[1] += solute ? 0.0 : sw * vq;
        } else {
          ec[1] = fma(sw, vc, ec[1]);
          eq[1] = fma(sw, vq, eq[1]);
        }
        if (DW) dwl += sw * seg;
        double gx, gy, gz;
        if constexpr (F32) {
          auto wide = [](double w) {
            float2 g;
            __builtin_memcpy(&g, &w, 8);
            return (double)g.x + (double)g.y;
          };
          gx = wide(W.gx[e]);
          gy = wide(W.gy[e]);
          gz = wide(W.gz[e]);
        } else {
          gx = W.gx[e];
          gy = W.gy[e];
          gz = W.gz[e];
        }
        // (unswitched pairs have no such term, also where two atoms coincide and their energy is not finite)
        const double v = dsw != 0.0 ? -dsw * (MODE == PAIR_REM ? vr : vc + vq) : 0.0;
        x3[0] = fma(v, gx, x3[0]);
        x3[1] = fma(v, gy, x3[1]);
        x3[2] = fma(v, gz, x3[2]);
        if (pass_st) {
          fsx = fma(v, gx, fsx);
          fsy = fma(v, gy, fsy);
          fsz = fma(v, gz, fsz);
          const double sx = shifted ? (double)W.sx[e] : 0.0, sy = shifted ? (double)W.sy[e] : 0.0,
                       sz = shifted ? (double)W.sz[e] : 0.0;
          const double fs[3] = {fsx, fsy, fsz}, sh3[3] = {sx, sy, sz};
#pragma unroll
          for (int k = 0; k < 9; ++k) st[k] = fma(-fs[k / 3], sh3[k % 3], st[k]);
        }
        shead = (shead + np) & (SLOT_RING - 1);
        ns -= np;
      }
      // ---- this batch's owner-atom forces: value 3 u + c on lanes 8 (3 u + c) ..
      double v[8];
#pragma unroll
      for (int h = 0; h < (3 * U + 7) / 8; ++h) {
        if (8 * h < 3 * nu) {
#pragma unroll
        for (int q = 0; q < 8; ++q) {
          const int w = 8 * h + q;
          v[q] = w < 3 * U ? fr[w < 3 * U ? w / 3 : 0][w % 3] : 0.0;
        }
        const double s = wave_sum8(v, buf, lane);
        const int w = 8 * h + (lane >> 3);
        if ((lane & 7) == 0 && w < 3 * nu) sh.fsum[wid][u0 + w / 3][w % 3] = s;
        }
      }
    }
  }
  // ---- energies, S'V vector and virial of the wave
  {
    double v[8] = {x3[0], x3[1], x3[2], ec[1], eq[1], DW ? dwl : 0.0, ec[0], eq[0]};
    const double s = wave_sum8(v, buf, lane);
    double *red = sh.red[wid];
    if (lane < PAIR_NACC) red[3 + lane] = 0.0;
    wave_lds_sync();
    if ((lane & 7) == 0) {
      // uconf / ucoul by typeij = typei + typej - 2 (0 slt-slt, 1 slt-slv, 2 slv-slv); both sides counted
      const int q = lane >> 3;
      if (q < 3) red[q] = s;
      else if (q == 3) red[3 + typei] = 0.5 * s;
      else if (q == 4) red[3 + 3 + typei] = 0.5 * s;
      else if (q == 5) red[3 + 15] = 0.5 * s;
      else if (q == 6) red[3 + typei - 1] = 0.5 * s;
      else red[3 + 3 + typei - 1] = 0.5 * s;
    }
    if (any_st) {
      const double s0 = wave_sum8(st, buf, lane);
      if ((lane & 7) == 0) red[3 + 6 + (lane >> 3)] = 0.5 * s0;
      const double s8 = wave_sum(st[8]);
      if (lane == 0) red[3 + 14] = 0.5 * s8;
    }
  }
  __syncthreads();
  // ---- owner-atom forces: the owner's waves in part order, then the S'V terms by mass fraction
  if (t < d.ngrp && part == 0) {
    double X[3] = {0.0, 0.0, 0.0}, f[3] = {0.0, 0.0, 0.0};
    for (int p = 0; p < S; ++p)
      for (int c = 0; c < 3; ++c) X[c] += sh.red[wid + p][c];
    if (lane < nI) {
      for (int p = 0; p < S; ++p)
        for (int c = 0; c < 3; ++c) f[c] += sh.fsum[wid + p][lane][c];
      const int a = ia0 + lane;
      const double gm = gmem(d.gmass)[a];
      const int pa = gmem(d.atomp)[a];
      const double cm[3] = {gmem(d.xpcm)[pa], gmem(d.ypcm)[pa], gmem(d.zpcm)[pa]};
      for (int c = 0; c < 3; ++c) f[c] += gm * X[c];
      gmem(d.fx)[a] = f[0];
      gmem(d.fy)[a] = f[1];
      gmem(d.fz)[a] = f[2];
      for (int c = 0; c < 3; ++c) {
        sh.fsum[wid][lane][c] = f[c];
        buf[3 * lane + c] = cm[c];
      }
    }
    wave_lds_sync();
    if (lane < 9) {  // the molecular virial F_a (x) C_a, in atom order
      double s = 0.0;
      for (int u = 0; u < nI; ++u) s += sh.fsum[wid][u][lane / 3] * buf[3 * u + lane % 3];
      sh.red[wid][3 + 6 + lane] += s;
    }
  }
  __syncthreads();
  if (threadIdx.x < PAIR_NACC) {
    double s = 0.0;
    for (int w = 0; w < PAIR_WAVES; ++w) s += sh.red[w][3 + threadIdx.x];
    gmem(d.part)[(size_t)blk * 16 + threadIdx.x] = s;
  }
}

// item l of nitems = nsys x nblkmax (system l / nblkmax), optionally XCD-grouped
__device__ __forceinline__ void pairs_item_index(int h, int nitems, int nblkmax, int remap, int &sys, int &blk) {
  const int l = remap ? xcd_remap(h, nitems) : h;
  sys = l / nblkmax;
  blk = l - sys * nblkmax;
}

// the item in its system's form: a plain system in a launch with alchemical ones
// gets what it gets alone
template <typename T, int MODE, int U>
__device__ __forceinline__ void pairs_form(const PairDesc &d, int blk, PairShared<U> &sh) {
  if constexpr (MODE == PAIR_ALCH) {
    if (!d.alch_pair) return pairs_item<T, PAIR_ANY, U>(d, blk, sh);
  }
  pairs_item<T, MODE, U>(d, blk, sh);
}

// W = minimum waves per SIMD the register allocation must allow (occupancy target)
template <typename T, int W, int MODE, int U>
__global__ void __launch_bounds__(256, W) k_pairs(const PairDesc *__restrict__ D, int remap) {
  __shared__ PairShared<U> sh;
  int sys, blk;
  pairs_item_index(blockIdx.x + gridDim.x * blockIdx.y, gridDim.x * gridDim.y, gridDim.x, remap, sys, blk);
  pairs_form<T, MODE, U>(D[sys], blk, sh);
}

// Persistent form: a fixed grid (a multiple of 8 workgroups, so each keeps to
// one XCD) walks all items of the batch with a grid stride.
template <typename T, int W, int MODE, int U>
__global__ void __launch_bounds__(256, W) k_pairs_persistent(const PairDesc *__restrict__ D, int remap, int nitems,
                                                             int nblkmax) {
  __shared__ PairShared<U> sh;
  for (int h = blockIdx.x; h < nitems; h += gridDim.x) {
    int sys, blk;
    pairs_item_index(h, nitems, nblkmax, remap, sys, blk);
    pairs_form<T, MODE, U>(D[sys], blk, sh);
    __syncthreads();
  }
}

template <typename T, int W, int MODE, int U>
static void launch_pair_kernel(bool persistent, dim3 grd, int g, hipStream_t st, const PairDesc *d_desc, int remap,
                               int nitems, int max_blk) {
  const dim3 blk(64 * PAIR_WAVES);
  if (persistent)
    hipLaunchKernelGGL((k_pairs_persistent<T, W, MODE, U>), dim3(g), blk, 0, st, d_desc, remap, nitems, max_blk);
  else
    hipLaunchKernelGGL((k_pairs<T, W, MODE, U>), grd, blk, 0, st, d_desc, remap);
}

__global__ void __launch_bounds__(1024) k_pairs_finalize(const PairDesc *__restrict__ D) {
  pairs_finalize(D[blockIdx.y], blockIdx.x);
}

// ================================================================ owner-atom loop form
//
// k_pairs_own: one wavefront per owner group, as k_pairs, with the roles of
// the loop and the lanes exchanged.  The lanes take the atoms of the
// neighbour groups (one atom each; whole groups packed into a pass of 64
// lanes) and loop over the owner group's atoms.  The owner atoms are the same
// across the wavefront and come through scalar loads; each lane loads its
// neighbour atom's record and LJ entries once per pass, and the pair loop
// touches no memory.  A list entry's group geometry, shell class and switch
// are computed once, when the entries are classified, and kept in LDS for
// the passes.  Each lane sums the owner atoms' forces in registers across the
// whole list (owner groups of at most OWN_REG atoms; systems with larger
// groups use k_pairs) and the wavefront reduces them at the end in a fixed
// order.
//
// Pair separations are the Cartesian group separation (image applied, FP64)
// plus the difference of the two atoms' Cartesian offsets from their group
// centres, so each pair costs three additions before its distance.

// (OWN_REG, the owner atoms whose force sums stay in registers: water, single atoms, is in kernels.hpp)

struct OwnWave {
  int ent[64];                  // the round's in-shell entries: neighbour group (sorted position)
  int pb[64];                   // half form: their first neighbour-side force slot
  int aoff[65];                 // exclusive prefix of their atom counts (aoff[n] = total)
  int nj[64];
  double gx[64], gy[64], gz[64];  // Cartesian separation of the group centres, image applied
  double sx[64], sy[64], sz[64];  // the image shift (reduced units)
  double sw[64], dsw[64];         // switch S and S'(r) / r of the group distance (1 and 0 unswitched)
};

struct OwnShared {
  OwnWave w[PAIR_WAVES];
  double red[PAIR_WAVES][PAIR_NACC];
};

template <typename T>
__device__ __forceinline__ void own_item(const PairDesc &d, int blk, OwnShared &sh) {
  if (blk >= d.nblk || !d.half) return;
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  OwnWave &W = sh.w[wid];
  // the owner group: wave-uniform, so its records come through scalar loads
  const int t = __builtin_amdgcn_readfirstlane(blk * PAIR_WAVES + wid);
  double fr[OWN_REG][3];
#pragma unroll
  for (int u = 0; u < OWN_REG; ++u) fr[u][0] = fr[u][1] = fr[u][2] = 0.0;
  double x3x = 0.0, x3y = 0.0, x3z = 0.0;  // the switched group pairs' S'(r) V vectors (owner side)
  double ec[2] = {0.0, 0.0}, eq[2] = {0.0, 0.0};  // LJ and Coulomb energy by the neighbour group's class
  double st[9];
#pragma unroll
  for (int k = 0; k < 9; ++k) st[k] = 0.0;
  int ia0 = 0, nI = 0, typei = 1, as0 = 0;
  if (t < d.ngrp) {
    const int4 gi = gload(d.sgi + t);
    as0 = gi.x;
    ia0 = gi.y;
    nI = gi.z & 255;
    typei = gi.z >> 8;
    const double4 gpi = gload(d.sgp + t);
    int nb0, nb1;
    if (d.nb_slab > 0) {
      nb0 = t * d.nb_slab;
      nb1 = nb0 + min(gmem(d.nb_cnt)[t], d.nb_slab);
    } else {
      nb0 = gmem(d.nb_off)[t];
      nb1 = gmem(d.nb_off)[t + 1];
    }
    for (int c0 = nb0; c0 < nb1; c0 += 64) {
      // ---- classify 64 entries; the in-shell ones are kept in list order
      const int jj = c0 + lane;
      const bool in = jj < nb1;
      const int tj = in ? gmem(d.nb_idx)[jj] : t;
      const GroupGeom gg = group_geom(gpi.x, gpi.y, gpi.z, gload_at(d.sgp, tj), d.co);
      const bool keep = in && in_shell(d, gg.drj);
      const int nJin = in ? (gload_at(d.sgi, tj).z & 255) : 0;
      const int nJ = keep ? nJin : 0;
      int mslot = -1;
      if (in) {
        // every forward entry's slots are written: the pair forces, or zeros outside the shell
        mslot = gmem(d.nb_mirror)[jj];
        if (!keep && mslot >= 0)
          for (int k = 0; k < nJin; ++k) {
            gmem(d.jpx)[mslot + k] = 0.0;
            gmem(d.jpy)[mslot + k] = 0.0;
            gmem(d.jpz)[mslot + k] = 0.0;
          }
      }
      const unsigned long long m = __ballot(keep);
      const int pos = __popcll(m & ((1ull << lane) - 1ull)), nc = __popcll(m);
      int incl = nJ;
#pragma unroll
      for (int off = 1; off < 64; off <<= 1) {
        const int y = __shfl_up(incl, off, 64);
        if (lane >= off) incl += y;
      }
      if (keep) {
        double sw = 1.0, dsw = 0.0;
        if (gg.drj >= d.r2out && gg.drj < d.r2out0) {
          const double rsp = sqrt(gg.drj);
          const double auxa = (d.arsout1 + 2.0 * rsp) / d.arsout2;
          const double auxb = d.rout0 - rsp;
          sw = auxa * (auxb * auxb);
          dsw = (-(2.0 * auxa * auxb) + 2.0 * (auxb * auxb) / d.arsout2) / rsp;
        } else if (gg.drj >= d.r2inn && gg.drj < d.r2inn0) {
          const double rsp = sqrt(gg.drj);
          const double auxa = (d.arsinn1 + 2.0 * rsp) / d.arsinn2;
          const double auxb = d.rinn0 - rsp;
          sw = 1.0 - auxa * (auxb * auxb);
          dsw = (2.0 * auxa * auxb - 2.0 * (auxb * auxb) / d.arsinn2) / rsp;
        }
        W.ent[pos] = tj;
        W.pb[pos] = mslot;
        W.aoff[pos] = incl - nJ;
        W.nj[pos] = nJ;
        W.gx[pos] = gg.xcc;
        W.gy[pos] = gg.ycc;
        W.gz[pos] = gg.zcc;
        W.sx[pos] = gg.sxm;
        W.sy[pos] = gg.sym;
        W.sz[pos] = gg.szm;
        W.sw[pos] = sw;
        W.dsw[pos] = dsw;
      }
      if (lane == 63) W.aoff[nc] = incl;
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
      __builtin_amdgcn_wave_barrier();
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
      // ---- passes: whole neighbour groups, one atom per lane
      for (int e0 = 0; e0 < nc;) {
        const int base = W.aoff[e0];
        const int ee = e0 + lane;
        const bool fits = ee < nc && W.aoff[ee] + W.nj[ee] - base <= 64;
        const int e1 = e0 + __popcll(__ballot(fits));
        // this lane's entry: the last e of the pass with aoff[e] - base <= lane
        int lo = e0, hi = e1;
        while (hi - lo > 1) {
          const int mid = (lo + hi) >> 1;
          if (W.aoff[mid] - base <= lane) lo = mid;
          else hi = mid;
        }
        const int e = lo, k = lane - (W.aoff[e] - base);
        const bool have = k < W.nj[e];
        const double xcc = W.gx[e], ycc = W.gy[e], zcc = W.gz[e];
        const double sw = have ? W.sw[e] : 0.0, dsw = have ? W.dsw[e] : 0.0;
        double fsx = 0.0, fsy = 0.0, fsz = 0.0;  // this lane's pair forces on the owner group
        double fbx = 0.0, fby = 0.0, fbz = 0.0;  // half form: the forces on this lane's neighbour atom
        double vc = 0.0, vq = 0.0;               // this lane's unswitched LJ and Coulomb energy
        int typej = 1, bs = 0, bo = 0, nJl = 0;
        bool fwd = false;
        int2 ib = make_int2(0, 0);
        AtomRec<T> rb = {T(0), T(0), T(0), T(0)};
        if (have) {
          const int4 gij = gload_at(d.sgi, W.ent[e]);
          typej = gij.z >> 8;
          fwd = true;  // a half list: this group is the lower one
          bs = gij.x + k;
          bo = gij.y + k;
          nJl = gij.z & 255;
          rb = atom_rec<T>(d, bs);
          ib = gload_at(d.sai, bs);
        }
        // separation = (owner centre - neighbour centre - image) + owner offset - neighbour offset
        const T bx = T(xcc - (double)rb.x), by = T(ycc - (double)rb.y), bz = T(zcc - (double)rb.z);
        const T swt = T(sw);
        if (have) {
          T c12[OWN_REG], c6[OWN_REG];
#pragma unroll
          for (int u = 0; u < OWN_REG; ++u) {
            c12[u] = T(0);
            c6[u] = T(0);
            if (u < nI) pair_lj<T>(d, gload(d.sai + as0 + u).x >> ATOM_FLAG_BITS, ib.x >> ATOM_FLAG_BITS, c12[u], c6[u]);
          }
#pragma unroll
          for (int u = 0; u < OWN_REG; ++u) {
            if (u >= nI) break;
            const AtomRec<T> ra = atom_rec<T>(d, as0 + u);
            const int2 ia = gload(d.sai + as0 + u);
            bool masked = false;
            if (ia.x & ib.x & ATOM_EX) masked = is_excluded(gmem(d.ex_off), gmem(d.ex_idx), ia0 + u, bo);
            if (d.any_heavy && !masked && !(gmem(d.mass)[bo] < d.massinfty || gmem(d.mass)[ia0 + u] < d.massinfty)) {
              // force.f:486-490: two atoms at or above massinfty are skipped only where the
              // list owner's atom has an exclusion partner in the other group (the owner
              // is the lower group: this one when fwd, the neighbour's otherwise)
              if (fwd)
                masked = (ia.x & ATOM_EX) && has_partner_in(gmem(d.ex_off), gmem(d.ex_idx), ia0 + u, bo - k, bo - k + nJl - 1);
              else
                masked = (ib.x & ATOM_EX) && has_partner_in(gmem(d.ex_off), gmem(d.ex_idx), bo, ia0, ia0 + nI - 1);
            }
            const T xc = bx + ra.x, yc = by + ra.y, zc = bz + ra.z;
            const T rsq = xc * xc + yc * yc + zc * zc;
            const T rinv = pair_rsqrt<T>(rsq);
            const T rsqi = rinv * rinv;
            const T r6 = rsqi * rsqi * rsqi;
            const T e6 = c6[u] * r6, e12 = c12[u] * r6 * r6;
            T conf = e12 - e6;
            T qforce = (T(12) * e12 - T(6) * e6) * rsqi;
            T cou = T(0);
            const T qq = ra.q * rb.q;
            if (!d.lskip_ewald) {
              const T rsp = rsq * rinv;
              const T alphar = T(d.alpha) * rsp;
              const T qt = pair_rcp<T>(T(1) + T(AS_QP) * alphar);
              const T expcst = pair_ewald_exp<T>(d, rsq, rsp);
              const T erfcst =
                  ((((T(AS_A5) * qt + T(AS_A4)) * qt + T(AS_A3)) * qt + T(AS_A2)) * qt + T(AS_A1)) * qt * expcst;
              cou = qq * erfcst * rinv;
              qforce += qq * (erfcst + T(d.twrtpi) * alphar * expcst) * (rsqi * rinv);
            } else if (!d.ewald) {
              cou = qq * rinv;
              qforce += cou * rsqi;
            }
            if (masked) {
              conf = T(0);
              cou = T(0);
              qforce = T(0);
            }
            const T qf = qforce * swt;
            const double fx = (double)(qf * xc), fy = (double)(qf * yc), fz = (double)(qf * zc);
            fr[u][0] += fx;
            fr[u][1] += fy;
            fr[u][2] += fz;
            fsx += fx;
            fsy += fy;
            fsz += fz;
            fbx -= fx;
            fby -= fy;
            fbz -= fz;
            vc += (double)conf;
            vq += (double)cou;
          }
        }
        // energies: each pair once (the j > i direction), scaled by the switch
        if (fwd) {
          ec[typej - 1] += sw * vc;
          eq[typej - 1] += sw * vq;
        }
        // S'(r) V of switched group pairs (force.f:756-817), V the group pair's
        // unswitched energy summed over the neighbour group's lanes
        double x3 = 0.0, y3 = 0.0, z3 = 0.0;
        if (__ballot(dsw != 0.0)) {
          const double v = vc + vq;
          const int first = lane - k;
          const int njl = have ? W.nj[e] : 0;
          double cmt = 0.0;
          for (int u = 0; u < d.max_group; ++u) {
            const double o = __shfl(v, (first + u) & 63, 64);
            if (u < njl) cmt += o;
          }
          x3 = -(dsw * cmt * xcc);
          y3 = -(dsw * cmt * ycc);
          z3 = -(dsw * cmt * zcc);
          if (have && k == 0) {
            x3x += x3;
            x3y += y3;
            x3z += z3;
          }
          if (have && dsw != 0.0) {
            // the neighbour group's share, -x3 by its atoms' mass fractions
            const double mb = gmem(d.gmass)[bo];
            fbx -= mb * x3;
            fby -= mb * y3;
            fbz -= mb * z3;
          }
        }
        if (have) {
          const int slot = W.pb[e];
          if (slot >= 0) {
            gmem(d.jpx)[slot + k] = fbx;
            gmem(d.jpy)[slot + k] = fby;
            gmem(d.jpz)[slot + k] = fbz;
          }
        }
        // molecular virial: the image-shift terms of pairs across the cell boundary
        if (fwd) {
          const double sxm = W.sx[e], sym = W.sy[e], szm = W.sz[e];
          if (sxm != 0.0 || sym != 0.0 || szm != 0.0) {
            if (k == 0) {
              fsx += x3;
              fsy += y3;
              fsz += z3;
            }
            st[0] -= fsx * sxm; st[1] -= fsx * sym; st[2] -= fsx * szm;
            st[3] -= fsy * sxm; st[4] -= fsy * sym; st[5] -= fsy * szm;
            st[6] -= fsz * sxm; st[7] -= fsz * sym; st[8] -= fsz * szm;
          }
        }
        e0 = e1;
      }
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
      __builtin_amdgcn_wave_barrier();
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    }
  }
  // ---- owner-atom forces: lane sums in lane order, then the S'V terms by mass fraction
  if (t < d.ngrp) {
    const double X = wave_sum(x3x), Y = wave_sum(x3y), Z = wave_sum(x3z);
    double fxa = 0.0, fya = 0.0, fza = 0.0;
#pragma unroll
    for (int u = 0; u < OWN_REG; ++u) {
      if (u < nI) {
        const double sx = wave_sum(fr[u][0]), sy = wave_sum(fr[u][1]), sz = wave_sum(fr[u][2]);
        if (lane == u) {
          fxa = sx;
          fya = sy;
          fza = sz;
        }
      }
    }
    if (lane < nI) {
      const int a = ia0 + lane;
      const double ma = gmem(d.gmass)[a];
      fxa += ma * X;
      fya += ma * Y;
      fza += ma * Z;
      gmem(d.fx)[a] = fxa;
      gmem(d.fy)[a] = fya;
      gmem(d.fz)[a] = fza;
      // (k_pairs_jsum adds the molecular virial once the neighbour-side forces are in)
    }
  }
  // ---- energies and virial: wave, then block, fixed order
  double vals[PAIR_NACC];
#pragma unroll
  for (int k = 0; k < PAIR_NACC; ++k) vals[k] = 0.0;
  // uconf / ucoul by typeij = typei + typej - 2 (0 slt-slt, 1 slt-slv, 2 slv-slv)
  vals[typei - 1] = ec[0];
  vals[typei] = ec[1];
  vals[3 + typei - 1] = eq[0];
  vals[3 + typei] = eq[1];
#pragma unroll
  for (int k = 0; k < 9; ++k) vals[6 + k] = st[k];
#pragma unroll
  for (int k = 0; k < PAIR_NACC; ++k) {
    const double v = wave_sum(vals[k]);
    if (lane == 0) sh.red[wid][k] = v;
  }
  __syncthreads();
  if (threadIdx.x < PAIR_NACC) {
    double s = 0.0;
    for (int w = 0; w < PAIR_WAVES; ++w) s += sh.red[w][threadIdx.x];
    gmem(d.part)[(size_t)blk * 16 + threadIdx.x] = s;
  }
}

template <typename T, int W>
__global__ void __launch_bounds__(256, W) k_pairs_own(const PairDesc *__restrict__ D, int remap) {
  __shared__ OwnShared sh;
  int sys, blk;
  pairs_item_index(blockIdx.x + gridDim.x * blockIdx.y, gridDim.x * gridDim.y, gridDim.x, remap, sys, blk);
  own_item<T>(D[sys], blk, sh);
}

template <typename T, int W>
__global__ void __launch_bounds__(256, W) k_pairs_own_persistent(const PairDesc *__restrict__ D, int remap,
                                                                 int nitems, int nblkmax) {
  __shared__ OwnShared sh;
  for (int h = blockIdx.x; h < nitems; h += gridDim.x) {
    int sys, blk;
    pairs_item_index(h, nitems, nblkmax, remap, sys, blk);
    own_item<T>(D[sys], blk, sh);
    __syncthreads();
  }
}

template <typename T, int W>
static void launch_own_kernel(bool persistent, dim3 grd, int g, hipStream_t st, const PairDesc *d_desc, int remap,
                              int nitems, int max_blk) {
  const dim3 blk(64 * PAIR_WAVES);
  if (persistent)
    hipLaunchKernelGGL((k_pairs_own_persistent<T, W>), dim3(g), blk, 0, st, d_desc, remap, nitems, max_blk);
  else
    hipLaunchKernelGGL((k_pairs_own<T, W>), grd, blk, 0, st, d_desc, remap);
}

// Half form, after the pair kernel: each group's atoms add the neighbour-side
// forces of its reverse entries (one wavefront per group, lanes over
// (reverse entry, atom) in memory order, lane sums combined in lane order),
// then the molecular virial sum F_a (x) C_a of the total forces.
__global__ void __launch_bounds__(256) k_pairs_jsum(const PairDesc *__restrict__ D) {
  __shared__ double red[PAIR_WAVES][64][3];
  __shared__ double vir[PAIR_WAVES][9];
  const PairDesc &d = D[blockIdx.y];
  const int blk = blockIdx.x;
  if (blk >= d.nblk || !d.half) return;
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  const int t = __builtin_amdgcn_readfirstlane(blk * PAIR_WAVES + wid);
  double st[9];
#pragma unroll
  for (int k = 0; k < 9; ++k) st[k] = 0.0;
  if (t < d.ngrp) {
    const int4 gi = gload(d.sgi + t);
    const int ia0 = gi.y, nI = gi.z & 255;
    int nr = min(gmem(d.nb_rcount)[t], d.nb_slab);
    const int base = gmem(d.nb_rbase)[t];
    if (base < 0 || (long long)base + (long long)nr * nI > d.pcap) nr = 0;  // an overflowed build (flagged)
    const int nrc = 64 / nI, rc = lane / nI, k = lane - rc * nI;
    double sx = 0.0, sy = 0.0, sz = 0.0;
    if (rc < nrc)
      for (int r = rc; r < nr; r += nrc) {
        const int idx = base + r * nI + k;
        sx += gmem(d.jpx)[idx];
        sy += gmem(d.jpy)[idx];
        sz += gmem(d.jpz)[idx];
      }
    red[wid][lane][0] = sx;
    red[wid][lane][1] = sy;
    red[wid][lane][2] = sz;
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    if (lane < nI) {
      const int a = ia0 + lane;
      double fxa = gmem(d.fx)[a], fya = gmem(d.fy)[a], fza = gmem(d.fz)[a];
      for (int q = 0; q < nrc; ++q) {
        fxa += red[wid][q * nI + lane][0];
        fya += red[wid][q * nI + lane][1];
        fza += red[wid][q * nI + lane][2];
      }
      gmem(d.fx)[a] = fxa;
      gmem(d.fy)[a] = fya;
      gmem(d.fz)[a] = fza;
      const int pa = gmem(d.atomp)[a];
      const double cx = gmem(d.xpcm)[pa], cy = gmem(d.ypcm)[pa], cz = gmem(d.zpcm)[pa];
      st[0] = fxa * cx; st[1] = fxa * cy; st[2] = fxa * cz;
      st[3] = fya * cx; st[4] = fya * cy; st[5] = fya * cz;
      st[6] = fza * cx; st[7] = fza * cy; st[8] = fza * cz;
    }
  }
#pragma unroll
  for (int k = 0; k < 9; ++k) {
    const double v = wave_sum(st[k]);
    if (lane == 0) vir[wid][k] = v;
  }
  __syncthreads();
  if (threadIdx.x < 9) {
    double s = 0.0;
    for (int w = 0; w < PAIR_WAVES; ++w) s += vir[w][threadIdx.x];
    gmem(d.part2)[(size_t)blk * 9 + threadIdx.x] = s;
  }
}

int pair_split_for(int ngrp) {
  // ORAC_HIP_PAIR_SPLIT=1|2|4 overrides the choice for systems created after it is set
  const char *e = getenv("ORAC_HIP_PAIR_SPLIT");
  const int v = e ? atoi(e) : 0;
  if (v == 1 || v == 2 || v == 4) return v;
  (void)ngrp;
  return 1;  // extra waves per owner cost more than the tail they trim (24,460 atoms, 2: 92 us for 82)
}

// Occupancy target of k_pairs (plain form): on the 24.5k-atom system 4 waves
// per SIMD take 85 us in FP64 (4 registers spilled) and 3 take 96; FP32 fits
// 4.  The tuning value, then ORAC_HIP_PAIR_WAVES=2|3|4, override it.
template <typename T>
static int pair_occupancy(int tuned) {
  if (tuned == 2 || tuned == 3 || tuned == 4) return tuned;
  static int w = [] {
    const char *e = getenv("ORAC_HIP_PAIR_WAVES");
    int v = e ? atoi(e) : 4;
    return (v == 2 || v == 3 || v == 4) ? v : 4;
  }();
  return w;
}

// The half-list form (k_pairs_own) is selected by ORAC_HIP_PAIR_KERNEL=own,
// read when a resident system is created (its list layout); by default every
// system takes k_pairs on the full list.
// Measured on MI355X on the 24,460-atom system (one evaluation with a list
// rebuild): the half-list form's per-pair slots and its list build (split,
// reverse ranking, mirror search) cost more than the halved arithmetic saves
// (0.473 vs 0.192 ms in FP64, 0.390 vs 0.181 in FP32).
bool use_owner_kernel() {
  const char *e = getenv("ORAC_HIP_PAIR_KERNEL");
  return e && std::string(e) == "own";
}

template <typename T>
void check_pairs(const PairDesc *h, int nsys) {
  bool any_alch = false, any_rem = false;
  for (int s = 0; s < nsys; ++s) {
    if ((sizeof(T) == 4 && !h[s].sapf) || ((sizeof(T) == 8 || h[s].alch_pair) && !h[s].sapc))
      throw Error(E_STATE, "no atom records in this precision");
    if (h[s].half) {
      if (h[s].alch_pair || h[s].rematom || h[s].split != 1 || h[s].max_group > OWN_REG)
        throw Error(E_STATE, "half-list pair form on a system it does not serve");
      continue;
    }
    any_alch = any_alch || h[s].alch_pair != nullptr;
    any_rem = any_rem || h[s].rematom != nullptr;
    if (h[s].max_group > 64)
      throw Error(E_UNSUPPORTED, "groups larger than 64 atoms are not supported by the pair kernel");
  }
  if (any_alch && any_rem) throw Error(E_STATE, "alchemical and REM systems in one launch");
  if (any_rem && sizeof(T) == 4) throw Error(E_STATE, "REM pairs are evaluated in double precision");
}

template <typename T>
void launch_pairs(const PairDesc *d_desc, const PairDesc *h, int nsys, hipStream_t st, const Tuning &tu,
                  bool packed, bool finalize, hipEvent_t kbeg, hipEvent_t kend) {
  check_pairs<T>(h, nsys);
  int max_grp = 1, max_blk = 1;
  // half-list systems take the half form, the others k_pairs
  bool any_alch = false, any_rem = false, any_other = false, any_half = false;
  bool any_many = false, any_few = false;
  for (int s = 0; s < nsys; ++s) {
    // every system's groups are packed and its blocks launched, whichever form serves it
    max_grp = std::max(max_grp, h[s].ngrp);
    max_blk = std::max(max_blk, h[s].nblk);
    if (h[s].half) {
      any_half = true;
      continue;
    }
    any_many = any_many || h[s].many;
    any_few = any_few || !h[s].many;
    any_alch = any_alch || h[s].alch_pair != nullptr;
    any_rem = any_rem || h[s].rematom != nullptr;
    any_other = any_other || h[s].lskip_ewald || h[s].any_heavy || !h[s].lj_dense;
  }
  if (!packed) hipLaunchKernelGGL(k_pack_sorted, dim3((max_grp + 255) / 256, nsys), dim3(256), 0, st, d_desc);
  dim3 grd(max_blk, nsys);
  const int remap = tu.xcd_remap ? 1 : 0;
  const int waves = pair_occupancy<T>(tu.pair_waves);
  const int nitems = max_blk * nsys;
  if (kbeg) ORAC_HIP(hipEventRecord(kbeg, st));
  int g = 0;
  if (tu.persistent) {
    // CUs x workgroups per CU at the occupancy target (4 waves per workgroup)
    static int ncu = [] {
      int dev = 0, n = 0;
      if (hipGetDevice(&dev) != hipSuccess || hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) !=
                                                   hipSuccess)
        n = 256;
      return n > 0 ? n : 256;
    }();
    g = std::max(8, std::min(nitems, ncu * waves) / 8 * 8);
  }
  const bool pers = tu.persistent != 0;
  if (any_half) {
    switch (waves) {
      case 3: launch_own_kernel<T, 3>(pers, grd, g, st, d_desc, remap, nitems, max_blk); break;
      case 4: launch_own_kernel<T, 4>(pers, grd, g, st, d_desc, remap, nitems, max_blk); break;
      default: launch_own_kernel<T, 2>(pers, grd, g, st, d_desc, remap, nitems, max_blk); break;
    }
    hipLaunchKernelGGL(k_pairs_jsum, grd, dim3(64 * PAIR_WAVES), 0, st, d_desc);
  }
  // (the soft-core, REM and general forms at one occupancy target)
  auto full = [&](auto u) {
    constexpr int U = decltype(u)::value, W = U == OWN_MANY ? 2 : 3;
    if (any_alch) {
      launch_pair_kernel<T, W, PAIR_ALCH, U>(pers, grd, g, st, d_desc, remap, nitems, max_blk);
    } else if (any_rem) {
      if constexpr (sizeof(T) == 8)  // (check_pairs)
        launch_pair_kernel<T, W, PAIR_REM, U>(pers, grd, g, st, d_desc, remap, nitems, max_blk);
    } else if (any_other) {
      launch_pair_kernel<T, W, PAIR_ANY, U>(pers, grd, g, st, d_desc, remap, nitems, max_blk);
    } else if (U == OWN_MANY || waves < 3) {
      launch_pair_kernel<T, 2, PAIR_PLAIN, U>(pers, grd, g, st, d_desc, remap, nitems, max_blk);
    } else if constexpr (U == OWN_FEW) {
      if (waves == 3) launch_pair_kernel<T, 3, PAIR_PLAIN, U>(pers, grd, g, st, d_desc, remap, nitems, max_blk);
      else launch_pair_kernel<T, 4, PAIR_PLAIN, U>(pers, grd, g, st, d_desc, remap, nitems, max_blk);
    }
  };
  if (any_few) full(std::integral_constant<int, OWN_FEW>{});
  if (any_many) full(std::integral_constant<int, OWN_MANY>{});
  if (kend) ORAC_HIP(hipEventRecord(kend, st));
  if (finalize) hipLaunchKernelGGL(k_pairs_finalize, dim3(PAIR_NACC, nsys), dim3(1024), 0, st, d_desc);
}

template void check_pairs<double>(const PairDesc *, int);
template void check_pairs<float>(const PairDesc *, int);
template void launch_pairs<double>(const PairDesc *, const PairDesc *, int, hipStream_t, const Tuning &, bool, bool,
                                   hipEvent_t, hipEvent_t);
template void launch_pairs<float>(const PairDesc *, const PairDesc *, int, hipStream_t, const Tuning &, bool, bool,
                                  hipEvent_t, hipEvent_t);

}  // namespace orac
