// common.hpp -- shared device/host definitions of the ORAC nonbonded path on gfx950.
//
// Conventions (the reference's): reduced coordinates xp = oc.x with the box
// spanning [-1,1); co/oc/recip are 3x3 column-major (m[i + 3*j] = m(i+1,j+1));
// grids are Q(K1,K2,K3), K1 fastest; the half-complex grid is FQ(K1/2+1,K2,K3).
// Every kernel reads a descriptor array and takes its system from blockIdx.y,
// so one launch serves one system or a batch of replicas.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <stdexcept>
#include <string>

namespace orac {

struct Error : std::runtime_error {
  int code;
  Error(int c, const std::string &m) : std::runtime_error(m), code(c) {}
};

#define ORAC_HIP(call)                                                                             \
  do {                                                                                             \
    hipError_t e_ = (call);                                                                        \
    if (e_ != hipSuccess)                                                                          \
      throw ::orac::Error(3, std::string(#call " failed: ") + hipGetErrorString(e_));              \
  } while (0)

#define ORAC_REQUIRE(cond, code, msg)                                                              \
  do {                                                                                             \
    if (!(cond)) throw ::orac::Error((code), (msg));                                               \
  } while (0)

// status codes returned through the C ABI
enum Status { OK = 0, E_ARG = 1, E_CAPACITY = 2, E_HIP = 3, E_UNSUPPORTED = 4, E_STATE = 5 };

constexpr int MAX_ORDER = 8;       // B-spline order limit of the device kernels
constexpr int MAX_FFT_LEN = 256;   // longest pencil an FFT workgroup holds in LDS
constexpr int MAX_RADICES = 12;

// ---------------------------------------------------------------- PME

// Per-axis FFT plan: radix sequence and twiddle table tw[m] = exp(-2 pi i m / n).
struct FftAxis {
  int n;
  int nr;
  int radix[MAX_RADICES];
  const double2 *tw64;
  const float2 *tw32;
};

// One system's reciprocal-space state.
struct PmeDesc {
  int natoms;
  int K1, K2, K3, order;
  double recip[9];          // recip(i,j) = 0.5*oc(j,i)
  double volume, pi_f32, fac, rkcut2;
  double fixscale, fixinv;  // grid fixed point: value = int64 * fixinv
  const double *xp, *yp, *zp;   // reduced coordinates
  const double *co;             // 3x3 on device (cartesian = co . xp)
  const double *q;
  unsigned long long *Qfix;     // K1*K2*K3 int64 two's complement
  void *FQ;                     // complex half grid, double2 or float2
  void *Qr;                     // real grid after c2r, double or float
  const double *bsp1, *bsp2, *bsp3;
  FftAxis ax1, ax2, ax3;
  double *fx, *fy, *fz;         // PME forces
  int accumulate;               // 0: fx = f_pme, 1: fx += f_pme
  int tpx, tpy, tpz;            // pencils per FFT workgroup along K1, K2, K3
  int gx, gy;                   // workgroups of the K1 and K2 passes
  double *conv_part;            // per-block energy/virial partials [conv_nblk][8]
  int conv_nblk;                // workgroups of the K3 pass
  // molecular-virial correction (fft_pme.f:65-106)
  const int *atomp;             // 0-based molecule of each atom
  const double *xpcm, *ypcm, *zpcm;
  double *gather_part;          // per-block stc partials [nblk][9]
  int gather_nblk;
  // LDS-tiled spread: grid tiles of st1 x st2 x st3 points (st = 0: global-atomic spread)
  int st1, st2, st3, nb1, nb2, nb3;
  int *bin_cnt;                 // [nb1*nb2*nb3 + 1] atoms per tile bin; the last: atoms that found their bin full.
                                //   Zero before an evaluation (the forward FFT leaves them so)
  double4 *bin_fr;              // [nb1*nb2*nb3][bin_cap] {fr1, fr2, fr3, q} of each bin's atoms
  double4 *over_fr;             // [natoms] the same of the atoms beyond their bin's capacity
  int bin_cap;
  double bin_slots;             // slots allocated at bin_fr (0: not yet)
  int tiled;                    // 1: LDS-tiled spread, 0: global-atomic spread
  double *out;                  // [20]: eer, vir (3x3 col-major), stc1..stc9
  int energy_only;              // 1: spread, forward FFT and energy only (a lambda0 charge grid)
  double *fx_dst, *fy_dst, *fz_dst;  // when set, launch_tail adds fx/fy/fz into these
  const double *cfx, *cfy, *cfz;     // and then these (the system's correction forces), when set
};

// ---------------------------------------------------------------- helpers

// Global-memory view of a device pointer.  Pointers a kernel reads out of a
// descriptor are generic (flat) to the compiler; accesses through this view
// are global ones: no aperture check, a uniform base in SGPRs, and waits on
// the vector-memory counter only, so they overlap with LDS traffic.
template <typename T>
__device__ __forceinline__ __attribute__((address_space(1))) T *gmem(T *p) {
  return (__attribute__((address_space(1))) T *)p;
}

// HIP vector types (double4, int4, ...) through the global view: their
// member functions expect generic objects, so the native vector is moved.
template <typename V>
__device__ __forceinline__ V gload(const V *p) {
  typedef typename V::Native_vec_ N;
  const N n = *(__attribute__((address_space(1))) const N *)p;
  V v;
  __builtin_memcpy(&v, &n, sizeof(V));
  return v;
}
// Element i of an array of HIP vector types as a uniform base plus a 32-bit
// byte offset (i * sizeof(V) < 2^32), the form of a global load with a
// scalar base and one offset VGPR.
template <typename V>
__device__ __forceinline__ V gload_at(const V *base, unsigned i) {
  return gload(reinterpret_cast<const V *>(reinterpret_cast<const char *>(base) + (i * (unsigned)sizeof(V))));
}
template <typename V>
__device__ __forceinline__ void gstore(V *p, const V &v) {
  typedef typename V::Native_vec_ N;
  N n;
  __builtin_memcpy(&n, &v, sizeof(V));
  *(__attribute__((address_space(1))) N *)p = n;
}

__host__ __device__ inline int wrap_idx(int k0, int K) { return k0 >= 0 ? k0 : k0 + K; }

// Fortran ANINT/DNINT: round half away from zero.
__host__ __device__ inline double fnint(double x) { return round(x); }

// Cardinal B-spline weights and derivatives (Essmann recursion,
// pme_fftw3.f90:537-576): derivative taken before the last pass.
// 1 / (k - 1) for the passes k = 2..MAX_ORDER: the correctly rounded value,
// as the division gives it, in either precision
template <typename T>
__host__ __device__ inline T recip_km1(int k) {
  switch (k) {
    case 2: return T(1.0);
    case 3: return T(1.0 / 2.0);
    case 4: return T(1.0 / 3.0);
    case 5: return T(1.0 / 4.0);
    case 6: return T(1.0 / 5.0);
    case 7: return T(1.0 / 6.0);
    case 8: return T(1.0 / 7.0);
    default: return T(1) / T(k - 1);
  }
}

// (no contraction by the compiler: every caller, unrolled or not, gets the same
// weights bit for bit, with the sum fused on the device and each operation
// rounded on the host, as the reference's is)
template <typename T>
__host__ __device__ inline T bspline_term(T div, T w, int k, int j, T lo, T hi) {
#pragma clang fp contract(off)
#ifdef __HIP_DEVICE_COMPILE__
  return div * fma(w + T(j), lo, (T(k - j) - w) * hi);
#else
  return div * ((w + T(j)) * lo + (T(k - j) - w) * hi);
#endif
}

template <typename T>
__host__ __device__ inline void bspline_pass(T *c, T w, int k) {
#pragma clang fp contract(off)
  T div = recip_km1<T>(k);
  c[k - 1] = div * w * c[k - 2];
  for (int j = 1; j <= k - 2; ++j) c[k - j - 1] = bspline_term(div, w, k, j, c[k - j - 2], c[k - j - 1]);
  c[0] = div * (T(1) - w) * c[0];
}

template <typename T>
__host__ __device__ inline void fill_bspline(T w, int order, T *c, T *d) {
#pragma clang fp contract(off)
  c[order - 1] = T(0);
  c[1] = w;
  c[0] = T(1) - w;
  for (int k = 3; k <= order - 1; ++k) bspline_pass(c, w, k);
  d[0] = -c[0];
  for (int j = 2; j <= order; ++j) d[j - 1] = c[j - 2] - c[j - 1];
  bspline_pass(c, w, order);
}

// the same for an order known at compile time (the loops unroll, and the
// weights stay in registers)
template <typename T, int ORDER>
__device__ __forceinline__ void fill_bspline_n(T w, T *c, T *d) {
#pragma clang fp contract(off)
  c[ORDER - 1] = T(0);
  c[1] = w;
  c[0] = T(1) - w;
#pragma unroll
  for (int k = 3; k <= ORDER; ++k) {
    if (k == ORDER) {
      d[0] = -c[0];
#pragma unroll
      for (int j = 2; j <= ORDER; ++j) d[j - 1] = c[j - 2] - c[j - 1];
    }
    const T div = recip_km1<T>(k);
    c[k - 1] = div * w * c[k - 2];
#pragma unroll
    for (int j = 1; j <= ORDER - 2; ++j)
      if (j <= k - 2) c[k - j - 1] = bspline_term(div, w, k, j, c[k - j - 2], c[k - j - 1]);
    c[0] = div * (T(1) - w) * c[0];
  }
}

// 64-bit fixed point: round-to-nearest of v*scale, two's complement.
__device__ inline unsigned long long to_fix(double v, double scale) {
  return (unsigned long long)__double2ll_rn(v * scale);
}

template <typename T>
__device__ inline T wave_sum(T v) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
  return v;
}

// A wave's LDS writes above are read by its other lanes below.
__device__ __forceinline__ void wave_lds_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

__device__ __forceinline__ int lanes_below(unsigned long long m) {
  return __builtin_amdgcn_mbcnt_hi((unsigned)(m >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)m, 0u));
}

__device__ __forceinline__ double uniform(double v) {
  int w[2];
  __builtin_memcpy(w, &v, 8);
  w[0] = __builtin_amdgcn_readfirstlane(w[0]);
  w[1] = __builtin_amdgcn_readfirstlane(w[1]);
  __builtin_memcpy(&v, w, 8);
  return v;
}
__device__ __forceinline__ float uniform(float v) {
  return __int_as_float(__builtin_amdgcn_readfirstlane(__float_as_int(v)));
}
__device__ __forceinline__ int uniform(int v) { return __builtin_amdgcn_readfirstlane(v); }

// Quotient of a small index (below 2^20) by a runtime divisor (below 2^11): the
// float quotient of the half-shifted index is off by less than 2^-2 / d, so its
// floor is exact, in three instructions rather than an integer division.
struct FastDiv {
  int d;
  float inv;
  __device__ __forceinline__ explicit FastDiv(int n) : d(n), inv(1.0f / (float)n) {}
  __device__ __forceinline__ int div(int x) const { return (int)(((float)x + 0.5f) * inv); }
  __device__ __forceinline__ int div(int x, int &rem) const {
    const int q = div(x);
    rem = x - q * d;
    return q;
  }
};

// Sum over a 1024-thread workgroup in fixed order, to every thread.
__device__ inline double block_sum_1024(double v) {
  __shared__ double red[16];
  v = wave_sum(v);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
  __syncthreads();
  double s = 0.0;
#pragma unroll
  for (int w = 0; w < 16; ++w) s += red[w];
  return s;
}

// Exclusive prefix sum of in[0..n) into out (may be in; both 16-byte aligned) by
// one 1024-thread workgroup; returns the total to every thread.  Each wavefront
// takes a contiguous part of up to SCAN_ROWS rows of 64 x 4, all of them loaded
// before the first sum, so the scan waits for memory once per 16,384 elements:
// the 27,001 cells of 103k atoms take 14 us (5 alone) where threads of contiguous parts,
// one dependent load after the other and no two lanes in one line, took 38.
constexpr int SCAN_ROWS = 4;
__device__ inline int block_exclusive_scan(const int *in, int *out, int n) {
  __shared__ int wsum[16];
  const int lane = threadIdx.x & 63, wid = uniform((int)(threadIdx.x >> 6));
  int done = 0;
  for (int i0 = 0; i0 < n; i0 += 4096 * SCAN_ROWS) {
    const int rows = min(SCAN_ROWS, (n - i0 + 4095) >> 12), j0 = i0 + wid * 256 * rows + 4 * lane;
    int4 v[SCAN_ROWS];
    int s = 0;
#pragma unroll
    for (int r = 0; r < SCAN_ROWS; ++r) {
      const int j = j0 + 256 * r;
      v[r] = make_int4(0, 0, 0, 0);
      if (r >= rows) continue;
      if (j + 3 < n) v[r] = gload(reinterpret_cast<const int4 *>(in + j));
      else {
        if (j < n) v[r].x = gmem(in)[j];
        if (j + 1 < n) v[r].y = gmem(in)[j + 1];
        if (j + 2 < n) v[r].z = gmem(in)[j + 2];
      }
    }
#pragma unroll
    for (int r = 0; r < SCAN_ROWS; ++r) s += v[r].x + v[r].y + v[r].z + v[r].w;
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) s += __shfl_xor(s, off, 64);
    if (lane == 0) wsum[wid] = s;
    __syncthreads();
    int run = done;
#pragma unroll
    for (int w = 0; w < 16; ++w) {
      const int x = wsum[w];
      run += w < wid ? x : 0;
      done += x;
    }
#pragma unroll
    for (int r = 0; r < SCAN_ROWS; ++r) {
      if (r >= rows) continue;
      const int j = j0 + 256 * r, sum = v[r].x + v[r].y + v[r].z + v[r].w;
      int x = sum;
#pragma unroll
      for (int off = 1; off < 64; off <<= 1) {
        const int y = __shfl_up(x, off, 64);
        if (lane >= off) x += y;
      }
      int4 o;
      o.x = run + x - sum;
      o.y = o.x + v[r].x;
      o.z = o.y + v[r].y;
      o.w = o.z + v[r].z;
      if (j + 3 < n) gstore(reinterpret_cast<int4 *>(out + j), o);
      else {
        if (j < n) gmem(out)[j] = o.x;
        if (j + 1 < n) gmem(out)[j + 1] = o.y;
        if (j + 2 < n) gmem(out)[j + 2] = o.z;
      }
      run += __builtin_amdgcn_readlane(x, 63);
    }
    __syncthreads();  // every thread has read wsum before it is written again
  }
  return done;
}

// Fractional grid coordinate along one reciprocal axis (pme_fftw3.f90:151-160).
__device__ inline double frac_coord(double x, double y, double z, const double *recip, int col, int K) {
  double w = x * recip[3 * col] + y * recip[3 * col + 1] + z * recip[3 * col + 2];
  return K * (w - fnint(w) + 0.5);
}

__device__ inline void cartesian(const double *co, double xp, double yp, double zp, double &x, double &y, double &z) {
  x = co[0] * xp + co[3] * yp + co[6] * zp;
  y = co[1] * xp + co[4] * yp + co[7] * zp;
  z = co[2] * xp + co[5] * yp + co[8] * zp;
}

// atom a (whole wavefronts; a at or past natoms: none) into its spread tile's bin
__device__ inline void bin_atom(const PmeDesc &d, int a) {
  const int lane = threadIdx.x & 63;
  int bin = -1;
  double4 f = make_double4(0.0, 0.0, 0.0, 0.0);
  if (a < d.natoms) {
    double x, y, z;
    cartesian(d.co, gmem(d.xp)[a], gmem(d.yp)[a], gmem(d.zp)[a], x, y, z);
    double fr1 = frac_coord(x, y, z, d.recip, 0, d.K1);
    double fr2 = frac_coord(x, y, z, d.recip, 1, d.K2);
    double fr3 = frac_coord(x, y, z, d.recip, 2, d.K3);
    // (non-finite coordinates are not spread)
    if (fr1 >= 0.0 && fr1 <= d.K1 && fr2 >= 0.0 && fr2 <= d.K2 && fr3 >= 0.0 && fr3 <= d.K3) {
      // fr = K (w - anint(w) = 0.5 exactly) is the grid origin: same spline weights
      if (fr1 >= d.K1) fr1 -= d.K1;
      if (fr2 >= d.K2) fr2 -= d.K2;
      if (fr3 >= d.K3) fr3 -= d.K3;
      f = make_double4(fr1, fr2, fr3, gmem(d.q)[a]);
      bin = (int)fr1 / d.st1 + d.nb1 * ((int)fr2 / d.st2 + d.nb2 * ((int)fr3 / d.st3));
    }
  }
  // Neighbouring atoms fall in the same tile: the lanes of one bin are counted
  // by one atomic of their lowest lane, all bins' atomics in flight together.
  unsigned long long todo = __ballot(bin >= 0), mine = 0ull;
  while (todo) {  // the same on every lane of the wavefront
    const int lb = __builtin_amdgcn_readlane(bin, __ffsll((long long)todo) - 1);
    const unsigned long long same = __ballot(bin == lb);
    if (bin == lb) mine = same;
    todo &= ~same;
  }
  if (bin < 0) mine = 1ull << lane;
  const int leader = __ffsll((long long)mine) - 1;
  int base = 0;
  if (bin >= 0 && lane == leader) base = atomicAdd(&d.bin_cnt[bin], __popcll(mine));
  base = __shfl(base, leader, 64);
  if (bin < 0) return;
  const int pos = base + __popcll(mine & ((1ull << lane) - 1ull));
  if (pos < d.bin_cap) {
    gstore(d.bin_fr + (size_t)bin * d.bin_cap + pos, f);
    return;
  }
  // the wavefront's atoms beyond their bins' room: one atomic on the list's count
  const unsigned long long over = __ballot(1);
  const int first = __ffsll((long long)over) - 1;
  int at = 0;
  if (lane == first) at = atomicAdd(&d.bin_cnt[d.nb1 * d.nb2 * d.nb3], __popcll(over));
  at = __builtin_amdgcn_readlane(at, first) + lanes_below(over);
  gstore(d.over_fr + at, f);
}

// lane J of each group of four lanes, to all four
template <int J>
__device__ __forceinline__ double quad_bcast(double v) {
  int w[2];
  __builtin_memcpy(w, &v, 8);
#pragma unroll
  for (int k = 0; k < 2; ++k) w[k] = __builtin_amdgcn_update_dpp(0, w[k], J * 0x55, 0xf, 0xf, true);
  __builtin_memcpy(&v, w, 8);
  return v;
}

// d.out[20]: eer, vir(3x3 col-major), stc(3x3 row-major as stc1..stc9).  A
// 1024-thread workgroup reduces one component in fixed order: k < 7 the
// convolution partials (scalar_sum.f:125-133 halving and symmetrisation),
// k >= 7 the molecular-virial partials.
__device__ inline void pme_finalize(const PmeDesc &d, int k) {
  if (k >= 7 && d.energy_only) {  // no gather: no molecular-virial terms
    if (threadIdx.x == 0) d.out[10 + (k - 7)] = 0.0;
    return;
  }
  const double *src = k < 7 ? d.conv_part + k : d.gather_part + (k - 7);
  const int nrow = k < 7 ? d.conv_nblk : d.gather_nblk, stride = k < 7 ? 8 : 9;
  double s = 0.0;
#pragma unroll 4
  for (int r = threadIdx.x; r < nrow; r += 1024) s += gmem(src)[(size_t)r * stride];
  s = block_sum_1024(s);
  if (threadIdx.x != 0) return;
  double *o = d.out;
  switch (k) {
    case 0: o[0] = 0.5 * s; break;
    case 1: o[1] = 0.5 * s; break;
    case 2: o[5] = 0.5 * s; break;
    case 3: o[9] = 0.5 * s; break;
    case 4: o[4] = o[2] = 0.5 * s; break;  // vir(1,2) = vir(2,1)
    case 5: o[7] = o[3] = 0.5 * s; break;  // vir(1,3) = vir(3,1)
    case 6: o[8] = o[6] = 0.5 * s; break;  // vir(2,3) = vir(3,2)
    default: o[10 + (k - 7)] = s; break;
  }
}

// The reciprocal forces of a system evaluated beside its direct sum are
// written to their own arrays; atom a's are added to its direct force once
// both are done, and then the corrections.
__device__ inline void pme_combine(const PmeDesc &d, int a) {
  if (!d.fx_dst || a >= d.natoms) return;
  double x = gmem(d.fx_dst)[a] + gmem(d.fx)[a], y = gmem(d.fy_dst)[a] + gmem(d.fy)[a],
         z = gmem(d.fz_dst)[a] + gmem(d.fz)[a];
  if (d.cfx) {
    x += gmem(d.cfx)[a];
    y += gmem(d.cfy)[a];
    z += gmem(d.cfz)[a];
  }
  gmem(d.fx_dst)[a] = x;
  gmem(d.fy_dst)[a] = y;
  gmem(d.fz_dst)[a] = z;
}

// Workgroups are dealt to the 8 XCDs round robin (hardware id h runs on XCD
// h % 8).  Mapping h to logical block (h % 8) * (n / 8) + h / 8 gives each XCD
// one contiguous range of logical blocks, so a system's blocks share an L2.
__device__ inline int xcd_remap(int h, int n) {
  const int q = n >> 3;
  if (h >= (q << 3)) return h;
  return (h & 7) * q + (h >> 3);
}

}  // namespace orac
