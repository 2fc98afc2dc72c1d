// pme.hip -- smooth PME reciprocal sum on gfx950.
//
// Stages (each one kernel, all systems of a batch in one launch via blockIdx.y):
//   k_spread      fractionals + order-p B-splines + charge spreading with
//                 64-bit fixed-point atomics (pme_fftw3.f90:132-163,234-298,487-576)
//   k_fft_plane_r2c  K3 planes: real rows along K1 -> half spectrum (FFTW r2c,
//                 pme_fftw3.f90:114), then K2; per axis for large planes:
//   k_fft_x_r2c, k_fft_pencil
//   k_fft_z_conv  pencils along K3: forward FFT, influence function with
//                 energy and virial (scalar_sum.f:1-135), inverse FFT, in LDS
//   k_fft_plane_c2r (k_fft_pencil, k_fft_x_c2r)  back: K2, then half spectrum
//                 -> real rows (FFTW c2r, pme_fftw3.f90:116)
//   k_gather      forces from the convolved grid (pme_fftw3.f90:311-372) and
//                 the molecular-virial correction terms (fft_pme.f:65-106)
//   k_pme_finalize fixed-order reduction of the per-block partials
// FFTs are LDS-staged mixed radix (2 to 6, 8) Stockham passes over tiles of
// pencils; loads and stores walk the contiguous K1 direction across threads.
#include "common.hpp"
#include "kernels.hpp"

namespace orac {

template <typename T>
struct cx {
  T x, y;
};
template <typename T>
__device__ inline cx<T> cmul(cx<T> a, cx<T> b) {
  return {a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x};
}
template <typename T>
__device__ inline cx<T> cadd(cx<T> a, cx<T> b) { return {a.x + b.x, a.y + b.y}; }
template <typename T>
__device__ inline cx<T> csub(cx<T> a, cx<T> b) { return {a.x - b.x, a.y - b.y}; }
template <typename T>
__device__ inline cx<T> cscale(cx<T> a, T s) { return {a.x * s, a.y * s}; }
// i*s*a for s = +-1
template <typename T, int S>
__device__ inline cx<T> cmuli(cx<T> a) { return S > 0 ? cx<T>{-a.y, a.x} : cx<T>{a.y, -a.x}; }

// the axis's twiddle table into LDS (one load per entry and workgroup)
template <typename T>
__device__ __forceinline__ void load_twiddles(cx<T> *tw, const FftAxis &ax) {
  for (int i = threadIdx.x; i < ax.n; i += blockDim.x) {
    if constexpr (sizeof(T) == 8) {
      const double2 w = gload(ax.tw64 + i);
      tw[i] = {w.x, w.y};
    } else {
      const float2 w = gload(ax.tw32 + i);
      tw[i] = {w.x, w.y};
    }
  }
}

// complex grid elements through the global view
__device__ __forceinline__ cx<double> cload(const cx<double> *p) {
  const double2 v = gload(reinterpret_cast<const double2 *>(p));
  return {v.x, v.y};
}
__device__ __forceinline__ cx<float> cload(const cx<float> *p) {
  const float2 v = gload(reinterpret_cast<const float2 *>(p));
  return {v.x, v.y};
}
__device__ __forceinline__ void cstore(cx<double> *p, cx<double> v) {
  gstore(reinterpret_cast<double2 *>(p), make_double2(v.x, v.y));
}
__device__ __forceinline__ void cstore(cx<float> *p, cx<float> v) {
  gstore(reinterpret_cast<float2 *>(p), make_float2(v.x, v.y));
}

template <typename T, int R, int S>
__device__ inline void dft(cx<T> *v) {
  if constexpr (R == 2) {
    cx<T> a = v[0], b = v[1];
    v[0] = cadd(a, b);
    v[1] = csub(a, b);
  } else if constexpr (R == 3) {
    const T s3 = T(0.8660254037844386467637231707529362);
    cx<T> t = cadd(v[1], v[2]), u = csub(v[1], v[2]);
    cx<T> a = csub(v[0], cscale(t, T(0.5)));
    cx<T> b = cmuli<T, S>(cscale(u, s3));
    v[0] = cadd(v[0], t);
    v[1] = cadd(a, b);
    v[2] = csub(a, b);
  } else if constexpr (R == 4) {
    cx<T> t0 = cadd(v[0], v[2]), t1 = csub(v[0], v[2]);
    cx<T> t2 = cadd(v[1], v[3]), t3 = cmuli<T, S>(csub(v[1], v[3]));
    v[0] = cadd(t0, t2);
    v[2] = csub(t0, t2);
    v[1] = cadd(t1, t3);
    v[3] = csub(t1, t3);
  } else if constexpr (R == 5) {
    const T c1 = T(0.3090169943749474241022934171828191), c2 = T(-0.8090169943749474241022934171828191);
    const T s1 = T(0.9510565162951535721164393333793821), s2 = T(0.5877852522924731291687059546390728);
    cx<T> t1 = cadd(v[1], v[4]), t2 = cadd(v[2], v[3]), t3 = csub(v[1], v[4]), t4 = csub(v[2], v[3]);
    cx<T> a1 = cadd(v[0], cadd(cscale(t1, c1), cscale(t2, c2)));
    cx<T> a2 = cadd(v[0], cadd(cscale(t1, c2), cscale(t2, c1)));
    cx<T> b1 = cmuli<T, S>(cadd(cscale(t3, s1), cscale(t4, s2)));
    cx<T> b2 = cmuli<T, S>(csub(cscale(t3, s2), cscale(t4, s1)));
    v[0] = cadd(v[0], cadd(t1, t2));
    v[1] = cadd(a1, b1);
    v[4] = csub(a1, b1);
    v[2] = cadd(a2, b2);
    v[3] = csub(a2, b2);
  } else if constexpr (R == 6) {
    // prime factors: input 3 n1 + 2 n2, output 3 k1 + 4 k2 (mod 6), and no twiddles between the
    // radix-2 and the radix-3 step, which in FP32 would round once more
    cx<T> s[3], d[3];
#pragma unroll
    for (int n = 0; n < 3; ++n) {
      const cx<T> p = v[2 * n], q = v[(2 * n + 3) % 6];
      s[n] = cadd(p, q);
      d[n] = csub(p, q);
    }
    dft<T, 3, S>(s);
    dft<T, 3, S>(d);
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      v[4 * k % 6] = s[k];
      v[(4 * k + 3) % 6] = d[k];
    }
  } else {  // 8: even and odd inputs, then one radix-2 step
    static_assert(R == 8);
    const T h = T(0.7071067811865475244);
    cx<T> e[4], o[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      e[k] = v[2 * k];
      o[k] = v[2 * k + 1];
    }
    dft<T, 4, S>(e);
    dft<T, 4, S>(o);
    o[1] = cmul(o[1], cx<T>{h, T(S) * h});
    o[2] = cmuli<T, S>(o[2]);
    o[3] = cmul(o[3], cx<T>{-h, T(S) * h});
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      v[k] = cadd(e[k], o[k]);
      v[k + 4] = csub(e[k], o[k]);
    }
  }
}

template <typename T, int R, int S>
__device__ __forceinline__ void stockham_pass(const cx<T> *a, cx<T> *b, int N, int LD, int TP, int Ns, const cx<T> *tw) {
  const FastDiv dNs(Ns), dNR(N / R);
  const int NR = dNR.d, twstep = FastDiv(Ns * R).div(N);
  for (int bi = threadIdx.x; bi < TP * NR; bi += blockDim.x) {
    int j, k;
    const int t = dNR.div(bi, j), jq = dNs.div(j, k);
    const cx<T> *src = a + t * LD;
    cx<T> *dst = b + t * LD;
    cx<T> v[R];
#pragma unroll
    for (int r = 0; r < R; ++r) v[r] = src[j + r * NR];
    if (Ns > 1) {
#pragma unroll
      for (int r = 1; r < R; ++r) {
        cx<T> w = tw[r * k * twstep];
        if (S > 0) w.y = -w.y;
        v[r] = cmul(v[r], w);
      }
    }
    dft<T, R, S>(v);
    const int idxD = jq * Ns * R + k;
#pragma unroll
    for (int r = 0; r < R; ++r) dst[idxD + r * Ns] = v[r];
  }
}

// TP pencils of length N, LD apart, held in LDS buffer a (b is scratch, tw the
// axis's twiddles in LDS); returns the buffer that holds the result.  Where
// lanes step from pencil to pencil, LD = N + 1 puts them in different banks.
template <typename T, int S>
__device__ __forceinline__ cx<T> *lds_fft(cx<T> *a, cx<T> *b, int N, int LD, int TP, const FftAxis &ax, const cx<T> *tw) {
  int Ns = 1;
  for (int p = 0; p < ax.nr; ++p) {
    int R = ax.radix[p];
    switch (R) {
      case 2: stockham_pass<T, 2, S>(a, b, N, LD, TP, Ns, tw); break;
      case 3: stockham_pass<T, 3, S>(a, b, N, LD, TP, Ns, tw); break;
      case 4: stockham_pass<T, 4, S>(a, b, N, LD, TP, Ns, tw); break;
      case 5: stockham_pass<T, 5, S>(a, b, N, LD, TP, Ns, tw); break;
      case 6: stockham_pass<T, 6, S>(a, b, N, LD, TP, Ns, tw); break;
      default: stockham_pass<T, 8, S>(a, b, N, LD, TP, Ns, tw); break;
    }
    __syncthreads();
    cx<T> *t = a;
    a = b;
    b = t;
    Ns *= R;
  }
  return a;
}

// ---------------------------------------------------------------- spread

__device__ inline int wrapK(int k0, int K) { return k0 < 0 ? k0 + K : (k0 >= K ? k0 - K : k0); }

// one thread per (atom, z-offset): order^2 fixed-point atomic adds
__global__ void __launch_bounds__(256) k_grid_zero(const PmeDesc *__restrict__ D) {
  const PmeDesc &d = D[blockIdx.y];
  if (d.tiled) return;
  const size_t G = (size_t)d.K1 * d.K2 * d.K3;
  for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < G; i += (size_t)gridDim.x * blockDim.x)
    d.Qfix[i] = 0ull;
}

template <typename T>
__global__ void __launch_bounds__(256) k_spread(const PmeDesc *__restrict__ D) {
  const PmeDesc &d = D[blockIdx.y];
  if (d.tiled) return;
  const int order = d.order;
  int tid = blockIdx.x * blockDim.x + threadIdx.x;
  int a = tid / order, i3 = tid - a * order;
  if (a >= d.natoms) return;
  double x, y, z;
  cartesian(d.co, d.xp[a], d.yp[a], d.zp[a], x, y, z);
  double fr1 = frac_coord(x, y, z, d.recip, 0, d.K1);
  double fr2 = frac_coord(x, y, z, d.recip, 1, d.K2);
  double fr3 = frac_coord(x, y, z, d.recip, 2, d.K3);
  // fr is in [0, K] for finite coordinates; anything else (NaN, inf) is skipped
  if (!(fr1 >= 0.0 && fr1 <= d.K1 && fr2 >= 0.0 && fr2 <= d.K2 && fr3 >= 0.0 && fr3 <= d.K3)) return;
  int b1 = (int)fr1, b2 = (int)fr2, b3 = (int)fr3;
  T th1[MAX_ORDER], th2[MAX_ORDER], th3[MAX_ORDER], dd[MAX_ORDER];
  fill_bspline<T>(T(fr1 - b1), order, th1, dd);
  fill_bspline<T>(T(fr2 - b2), order, th2, dd);
  fill_bspline<T>(T(fr3 - b3), order, th3, dd);
  // same product order as the tiled spread, th1 * (th2 * (th3 * q)), so both
  // paths put identical fixed-point values on the grid
  const T q3 = th3[i3] * T(d.q[a]);
  const int kk = wrapK(b3 - order + i3 + 1, d.K3);
  const double scale = d.fixscale;
  for (int i2 = 0; i2 < order; ++i2) {
    int jj = wrapK(b2 - order + i2 + 1, d.K2);
    T prod = th2[i2] * q3;
    size_t row = (size_t)d.K1 * (jj + (size_t)d.K2 * kk);
    for (int i1 = 0; i1 < order; ++i1) {
      int ii = wrapK(b1 - order + i1 + 1, d.K1);
      atomicAdd(&d.Qfix[row + ii], to_fix((double)(th1[i1] * prod), scale));
    }
  }
}

// ---------------------------------------------------------------- tiled spread
//
// Atoms are binned by the tile of their spline base point b = int(fr).  The
// tile (T1,T2,T3) of st1 x st2 x st3 grid points receives contributions from
// atoms with b in [t0, t0 + st + order - 2] per axis, i.e. from bins T and
// T + 1 (mod nb) when st >= order - 1 and st divides K.  One workgroup per
// tile accumulates those contributions in LDS with int64 atomics and stores
// its points: every grid point has one owner, no global atomics, no clearing,
// and sums of integers do not depend on their order.
//
// k_bin puts each atom straight into its bin's slots (fixed capacity, an
// overflow list beyond it), so no scan and no second pass over the atoms is
// needed: 20 + 5 + 6 us of counting, scanning and filling for 24,460 atoms
// became one kernel of 5.5 us.
// A resident evaluation bins in its preparing launch (k_prepare).
__global__ void __launch_bounds__(256) k_bin(const PmeDesc *__restrict__ D) {
  const PmeDesc &d = D[blockIdx.y];
  if (d.tiled) bin_atom(d, blockIdx.x * blockDim.x + threadIdx.x);
}

constexpr int SPREAD_TILE_MAX = 8;

// The tile-local range of an atom's stencil along one axis.  The stencil
// points are base + i, i = 0..order-1, base = b - order + 1 (+ K when the atom
// comes from the wrapped neighbour bin) minus the tile origin.  With two or
// more tiles along the axis (st >= order - 1) the points inside the tile are
// one range [ia, ib) and none of them wraps; with one tile (st = K) every
// point is inside after a wrap of the negative ones.
struct AxisRange {
  int l0, ia, ib, wrap;
};
__device__ inline AxisRange axis_range(int b, int order, int t0, int st, int K, int wrapped) {
  AxisRange r;
  r.l0 = b - order + 1 + (wrapped ? K : 0) - t0;
  if (st >= K) {
    r.ia = 0;
    r.ib = order;
    r.wrap = K;
  } else {
    r.ia = max(0, -r.l0);
    r.ib = min(order, st - r.l0);
    r.wrap = 0;
  }
  return r;
}

// k_spread_tile, in two alternating phases.  (1) One thread per candidate of
// the eight bins, taken as one flat sequence (a lookup in nine prefix sums),
// so the loads of all bins are in flight together; a candidate that reaches
// the tile writes its spline weights and tile-local ranges to LDS.  (2) The
// threads take (listed atom, z-plane, y-row) tasks and add a row's points.
// Bound by the latency of phase 1 and the LDS atomics of phase 2; 24,460 atoms on
// 64^3: 16 us, against 33 us when the bins were walked one after the other by
// (atom, plane) threads that re-read their weights from memory; 16 such systems
// in one launch 129 us against 344.  256 candidates a round keep the list within
// 64 KB of LDS at any order; 512 threads share its tasks (22 us with 256).  The tile is padded (st1 + 1,
// st2 + 1), which keeps z-planes and y-rows of one column on different banks.
constexpr int SPREAD_THREADS = 512, SPREAD_CAND = 256;  // threads; candidates per round
constexpr int SPREAD_TILE_WORDS = (SPREAD_TILE_MAX + 1) * (SPREAD_TILE_MAX + 1) * SPREAD_TILE_MAX;

// one listed atom: ranges (l0, ia | ib << 8 per axis), then 3 * order weights, the third times q
template <typename T>
__host__ __device__ constexpr int spread_rec_bytes(int order) {
  return 24 + ((3 * order * (int)sizeof(T) + 7) / 8) * 8;
}
template <typename T>
static size_t spread_lds_bytes(int order) {
  return (size_t)SPREAD_CAND * spread_rec_bytes<T>(order);
}

template <typename T, int ORDER>
__global__ void __launch_bounds__(SPREAD_THREADS) k_spread_tile(const PmeDesc *__restrict__ D) {
  extern __shared__ __align__(16) unsigned char list[];
  __shared__ unsigned long long tile[SPREAD_TILE_WORDS];
  __shared__ int pre[10], bins[8], listed;
  const PmeDesc &d = D[blockIdx.y];
  if (!d.tiled || (int)blockIdx.x >= d.nb1 * d.nb2 * d.nb3) return;
  const int order = ORDER > 0 ? ORDER : d.order;
  const int nb1 = d.nb1, nb2 = d.nb2, nb3 = d.nb3, cap = d.bin_cap;
  const int T1 = blockIdx.x % nb1, T2 = (blockIdx.x / nb1) % nb2, T3 = blockIdx.x / (nb1 * nb2);
  const int st1 = d.st1, st2 = d.st2, st3 = d.st3, P1 = st1 + 1, P2 = st2 + 1;
  const int t01 = T1 * st1, t02 = T2 * st2, t03 = T3 * st3;
  const int npts = st1 * st2 * st3;
  if (threadIdx.x < 8) {
    const int sb = threadIdx.x, o1 = sb & 1, o2 = (sb >> 1) & 1, o3 = sb >> 2;
    // with a single bin along an axis, the +1 neighbour is the same bin: visited once
    const bool skip = (o1 && nb1 == 1) || (o2 && nb2 == 1) || (o3 && nb3 == 1);
    const int B1 = T1 + o1 - (T1 + o1 >= nb1 ? nb1 : 0), B2 = T2 + o2 - (T2 + o2 >= nb2 ? nb2 : 0),
              B3 = T3 + o3 - (T3 + o3 >= nb3 ? nb3 : 0);
    const int bin = B1 + nb1 * (B2 + nb2 * B3);
    const int n = skip ? 0 : min(gmem(d.bin_cnt)[bin], cap);
    bins[sb] = bin;
    int x = n;
#pragma unroll
    for (int off = 1; off < 8; off <<= 1) {
      const int y = __shfl_up(x, off, 8);
      if (sb >= off) x += y;
    }
    pre[sb + 1] = x;
    if (sb == 0) pre[0] = 0;
    if (sb == 7) pre[9] = x + gmem(d.bin_cnt)[nb1 * nb2 * nb3];  // then the overflow list
  }
  if (threadIdx.x == 0) listed = 0;
  for (int i = threadIdx.x; i < P1 * P2 * st3; i += SPREAD_THREADS) tile[i] = 0ull;
  __syncthreads();
  const double scale = d.fixscale;
  const int in_bins = pre[8], total = pre[9], rec = spread_rec_bytes<T>(order);
  const FastDiv dO2(order * order), dO(order);
  for (int q0 = 0; q0 < total; q0 += SPREAD_CAND) {
    // ---- (1) candidates
    const int qi = q0 + threadIdx.x;
    if (qi < total && (int)threadIdx.x < SPREAD_CAND) {
      double4 f;
      if (qi < in_bins) {
        int sb = 0;
#pragma unroll
        for (int k = 1; k < 8; ++k) sb += pre[k] <= qi ? 1 : 0;
        f = gload(d.bin_fr + (size_t)bins[sb] * cap + (qi - pre[sb]));
      } else {
        f = gload(d.over_fr + (qi - in_bins));
      }
      const int b1 = (int)f.x, b2 = (int)f.y, b3 = (int)f.z;
      // the atom comes across the periodic boundary when its base point lies below the tile's origin
      const AxisRange x = axis_range(b1, order, t01, st1, d.K1, b1 < t01), y = axis_range(b2, order, t02, st2, d.K2, b2 < t02),
                      z = axis_range(b3, order, t03, st3, d.K3, b3 < t03);
      if (x.ia < x.ib && y.ia < y.ib && z.ia < z.ib) {
        unsigned char *rp = list + (size_t)atomicAdd(&listed, 1) * rec;
        int *ri = reinterpret_cast<int *>(rp);
        T *w = reinterpret_cast<T *>(rp + 24);
        ri[0] = x.l0;
        ri[1] = x.ia | x.ib << 8;
        ri[2] = y.l0;
        ri[3] = y.ia | y.ib << 8;
        ri[4] = z.l0;
        ri[5] = z.ia | z.ib << 8;
        constexpr int NO = ORDER > 0 ? ORDER : MAX_ORDER;
        T th[NO], dd[NO];
        const T qt = T(f.w);
        if constexpr (ORDER > 0) {
          fill_bspline_n<T, ORDER>(T(f.x - b1), th, dd);
#pragma unroll
          for (int i = 0; i < NO; ++i) w[i] = th[i];
          fill_bspline_n<T, ORDER>(T(f.y - b2), th, dd);
#pragma unroll
          for (int i = 0; i < NO; ++i) w[NO + i] = th[i];
          fill_bspline_n<T, ORDER>(T(f.z - b3), th, dd);
#pragma unroll
          for (int i = 0; i < NO; ++i) w[2 * NO + i] = th[i] * qt;
        } else {
          fill_bspline<T>(T(f.x - b1), order, th, dd);
          for (int i = 0; i < order; ++i) w[i] = th[i];
          fill_bspline<T>(T(f.y - b2), order, th, dd);
          for (int i = 0; i < order; ++i) w[order + i] = th[i];
          fill_bspline<T>(T(f.z - b3), order, th, dd);
          for (int i = 0; i < order; ++i) w[2 * order + i] = th[i] * qt;
        }
      }
    }
    __syncthreads();
    // ---- (2) rows
    const int ntask = listed * order * order;
    for (int task = threadIdx.x; task < ntask; task += SPREAD_THREADS) {
      int row, i2;
      const int at = dO2.div(task, row), i3 = dO.div(row, i2);
      const unsigned char *rp = list + (size_t)at * rec;
      const int *ri = reinterpret_cast<const int *>(rp);
      if (i3 < (ri[5] & 255) || i3 >= ri[5] >> 8 || i2 < (ri[3] & 255) || i2 >= ri[3] >> 8) continue;
      int lz = ri[4] + i3, ly = ri[2] + i2;
      if (lz < 0) lz += d.K3;  // (one tile along the axis: the only case with negative in-range points)
      if (ly < 0) ly += d.K2;
      const T *w = reinterpret_cast<const T *>(rp + 24);
      const T prod = w[order + i2] * w[2 * order + i3];
      unsigned long long *trow = tile + P1 * (ly + P2 * lz);
      const int l0 = ri[0], ia = ri[1] & 255, ib = ri[1] >> 8;
      if constexpr (ORDER > 0) {
#pragma unroll
        for (int i1 = 0; i1 < ORDER; ++i1) {
          int lx = l0 + i1;
          if (lx < 0) lx += d.K1;
          if (i1 >= ia && i1 < ib) atomicAdd(&trow[lx], to_fix((double)(w[i1] * prod), scale));
        }
      } else {
        for (int i1 = ia; i1 < ib; ++i1) {
          int lx = l0 + i1;
          if (lx < 0) lx += d.K1;
          atomicAdd(&trow[lx], to_fix((double)(w[i1] * prod), scale));
        }
      }
    }
    __syncthreads();
    if (threadIdx.x == 0) listed = 0;
    __syncthreads();
  }
  const FastDiv d1(st1), d2(st2);
  for (int i = threadIdx.x; i < npts; i += SPREAD_THREADS) {
    int lx, ly;
    const int yz = d1.div(i, lx), lz = d2.div(yz, ly);
    gmem(d.Qfix)[(size_t)(t01 + lx) + (size_t)d.K1 * ((t02 + ly) + (size_t)d.K2 * (t03 + lz))] =
        tile[lx + P1 * (ly + P2 * lz)];
  }
}

// tile edge along one axis: a divisor of K in [max(order - 1, 2), 8], the
// largest or the smallest; 0 if none
int spread_tile_edge(int K, int order, bool smallest) {
  const int lo = std::max(2, order - 1);
  if (smallest) {
    for (int s = lo; s <= SPREAD_TILE_MAX; ++s)
      if (K % s == 0) return s;
    return 0;
  }
  for (int s = SPREAD_TILE_MAX; s >= lo; --s)
    if (K % s == 0) return s;
  return 0;
}

// ---------------------------------------------------------------- transforms

// The transforms along K1 and K2 of one K3 plane in one workgroup, where two
// copies of the half spectrum and the twiddles fit its 160 KB of LDS.  Two real
// rows go through one complex transform; neither direction writes the plane
// between its axes.  Larger planes (100 x 100 in FP64, 144 x 144 in FP32) take
// a kernel per axis.  The three FFT launches with planes against the five
// without: 216 waters (FP64) 27 against 33 us, 24,460 atoms 45 against 49,
// 103k atoms (FP32, 108^3) 68 against 90, 16 systems of 24,460 114 against 190.
constexpr size_t PLANE_LDS = 160 * 1024;
__host__ __device__ inline int plane_buf(int K1, int K2) {
  const int rows = (K2 + 1) / 2 * (K1 + 1), cols = (K1 / 2 + 1) * (K2 + 1);
  return rows > cols ? rows : cols;
}
template <typename T>
__host__ __device__ inline size_t plane_lds(const PmeDesc &d) {
  return (2 * (size_t)plane_buf(d.K1, d.K2) + d.K1 + d.K2) * sizeof(cx<T>);
}
template <typename T>
__host__ __device__ inline bool use_planes(const PmeDesc &d) {
  return plane_lds<T>(d) <= PLANE_LDS;
}

template <typename T>
__global__ void __launch_bounds__(1024) k_fft_plane_r2c(const PmeDesc *__restrict__ D) {
  extern __shared__ __align__(16) unsigned char smem[];
  const PmeDesc &d = D[blockIdx.y];
  const int K1 = d.K1, K2 = d.K2, H = K1 / 2 + 1, P = (K2 + 1) / 2, LD1 = K1 + 1, LD2 = K2 + 1, z = blockIdx.x;
  if (z >= d.K3 || !use_planes<T>(d)) return;
  cx<T> *a = reinterpret_cast<cx<T> *>(smem), *b = a + plane_buf(K1, K2), *tw1 = b + plane_buf(K1, K2),
        *tw2 = tw1 + K1;
  const double inv = d.fixinv;
  const FastDiv dK1(K1), dH(H);
  const auto in = gmem(d.Qfix + (size_t)z * K1 * K2);
  load_twiddles(tw1, d.ax1);
  load_twiddles(tw2, d.ax2);
#pragma unroll 4
  for (int i = threadIdx.x; i < P * K1; i += blockDim.x) {
    int e;
    const int j = dK1.div(i, e);
    const long long q0 = (long long)in[(2 * j) * K1 + e], q1 = 2 * j + 1 < K2 ? (long long)in[(2 * j + 1) * K1 + e] : 0;
    a[j * LD1 + e] = {T((double)q0 * inv), T((double)q1 * inv)};
  }
  // the spread is done with its bins: empty for the next evaluation
  if (d.tiled)
    for (int i = z * blockDim.x + threadIdx.x; i <= d.nb1 * d.nb2 * d.nb3; i += d.K3 * blockDim.x)
      gmem(d.bin_cnt)[i] = 0;
  __syncthreads();
  cx<T> *r = lds_fft<T, -1>(a, b, K1, LD1, P, d.ax1, tw1), *s = r == a ? b : a;
  // rows 2j and 2j + 1 from their sum Z: (Z[k] + conj Z[-k]) / 2, (Z[k] - conj Z[-k]) / 2i
  for (int i = threadIdx.x; i < P * H; i += blockDim.x) {
    int k;
    const int j = dH.div(i, k);
    const cx<T> u = r[j * LD1 + k], w = r[j * LD1 + (k ? K1 - k : 0)];
    s[k * LD2 + 2 * j] = {T(0.5) * (u.x + w.x), T(0.5) * (u.y - w.y)};
    if (2 * j + 1 < K2) s[k * LD2 + 2 * j + 1] = {T(0.5) * (u.y + w.y), T(0.5) * (w.x - u.x)};
  }
  __syncthreads();
  r = lds_fft<T, -1>(s, r, K2, LD2, H, d.ax2, tw2);
  cx<T> *FQ = reinterpret_cast<cx<T> *>(d.FQ) + (size_t)z * K2 * H;
  for (int i = threadIdx.x; i < K2 * H; i += blockDim.x) {
    int k;
    const int y = dH.div(i, k);
    cstore(FQ + i, r[k * LD2 + y]);
  }
}

template <typename T>
__global__ void __launch_bounds__(1024) k_fft_plane_c2r(const PmeDesc *__restrict__ D) {
  extern __shared__ __align__(16) unsigned char smem[];
  const PmeDesc &d = D[blockIdx.y];
  const int K1 = d.K1, K2 = d.K2, H = K1 / 2 + 1, P = (K2 + 1) / 2, LD1 = K1 + 1, LD2 = K2 + 1, z = blockIdx.x;
  if (z >= d.K3 || d.energy_only || !use_planes<T>(d)) return;
  cx<T> *a = reinterpret_cast<cx<T> *>(smem), *b = a + plane_buf(K1, K2), *tw1 = b + plane_buf(K1, K2),
        *tw2 = tw1 + K1;
  const FastDiv dK1(K1), dH(H);
  const cx<T> *FQ = reinterpret_cast<const cx<T> *>(d.FQ) + (size_t)z * K2 * H;
  load_twiddles(tw1, d.ax1);
  load_twiddles(tw2, d.ax2);
#pragma unroll 4
  for (int i = threadIdx.x; i < K2 * H; i += blockDim.x) {
    int k;
    const int y = dH.div(i, k);
    a[k * LD2 + y] = cload(FQ + i);
  }
  __syncthreads();
  cx<T> *r = lds_fft<T, +1>(a, b, K2, LD2, H, d.ax2, tw2), *s = r == a ? b : a;
  // Z = X(row 2j) + i X(row 2j + 1), both Hermitian (the imaginary parts at 0 and K1 / 2 are not read)
  for (int i = threadIdx.x; i < P * H; i += blockDim.x) {
    int k;
    const int j = dH.div(i, k);
    cx<T> u = r[k * LD2 + 2 * j], w = {T(0), T(0)};
    if (2 * j + 1 < K2) w = r[k * LD2 + 2 * j + 1];
    if (k == 0 || 2 * k == K1) u.y = w.y = T(0);
    s[j * LD1 + k] = {u.x - w.y, u.y + w.x};
    if (k > 0 && K1 - k >= H) s[j * LD1 + K1 - k] = {u.x + w.y, w.x - u.y};
  }
  __syncthreads();
  r = lds_fft<T, +1>(s, r, K1, LD1, P, d.ax1, tw1);
  T *Qr = reinterpret_cast<T *>(d.Qr) + (size_t)z * K2 * K1;
  for (int i = threadIdx.x; i < K2 * K1; i += blockDim.x) {
    int e;
    const int y = dK1.div(i, e);
    const cx<T> v = r[(y >> 1) * LD1 + e];
    gmem(Qr)[i] = y & 1 ? v.y : v.x;
  }
}

constexpr int CONV_PTS = 8;  // grid points per thread of k_fft_z_conv at most

// Rows along K1: fixed-point grid -> half spectrum.  TP rows per block.
template <typename T>
__global__ void __launch_bounds__(256) k_fft_x_r2c(const PmeDesc *__restrict__ D) {
  extern __shared__ __align__(16) unsigned char smem[];
  const PmeDesc &d = D[blockIdx.y];
  const int N = d.K1, H = N / 2 + 1, rows = d.K2 * d.K3, TP = d.tpx;
  if ((int)blockIdx.x >= d.gx || use_planes<T>(d)) return;
  cx<T> *a = reinterpret_cast<cx<T> *>(smem);
  cx<T> *b = a + TP * N;
  cx<T> *tw = b + TP * N;
  const int row0 = blockIdx.x * TP;
  const double inv = d.fixinv;
  const FastDiv dN(N), dH(H);
  load_twiddles(tw, d.ax1);
  for (int i = threadIdx.x; i < TP * N; i += blockDim.x) {
    int e;
    const int row = row0 + dN.div(i, e);
    T v = T(0);
    if (row < rows) v = T((double)(long long)gmem(d.Qfix)[(size_t)row * N + e] * inv);
    a[i] = {v, T(0)};
  }
  // the spread is done with its bins: empty for the next evaluation
  if (d.tiled)
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i <= d.nb1 * d.nb2 * d.nb3; i += d.gx * blockDim.x)
      gmem(d.bin_cnt)[i] = 0;
  __syncthreads();
  cx<T> *r = lds_fft<T, -1>(a, b, N, N, TP, d.ax1, tw);
  cx<T> *FQ = reinterpret_cast<cx<T> *>(d.FQ);
  for (int i = threadIdx.x; i < TP * H; i += blockDim.x) {
    int e;
    const int t = dH.div(i, e), row = row0 + t;
    if (row < rows) cstore(FQ + (size_t)row * H + e, r[t * N + e]);
  }
}

// Complex pencils along K2 of the half grid: pencil p has base (p % H) +
// (p / H) * H * K2 and element stride H.
template <typename T, int S>
__global__ void __launch_bounds__(256) k_fft_pencil(const PmeDesc *__restrict__ D) {
  extern __shared__ __align__(16) unsigned char smem[];
  const PmeDesc &d = D[blockIdx.y];
  const int H = d.K1 / 2 + 1, TP = d.tpy;
  if ((int)blockIdx.x >= d.gy || (S > 0 && d.energy_only) || use_planes<T>(d)) return;
  const FftAxis &ax = d.ax2;
  const int N = ax.n, npen = H * d.K3;
  const size_t S1 = (size_t)H * d.K2, Se = (size_t)H;
  const int p0 = blockIdx.x * TP;
  if (p0 >= npen) return;
  cx<T> *a = reinterpret_cast<cx<T> *>(smem);
  cx<T> *b = a + TP * N;
  cx<T> *FQ = reinterpret_cast<cx<T> *>(d.FQ);
  cx<T> *tw = b + TP * N;
  const FastDiv dTP(TP), dH(H);
  load_twiddles(tw, ax);
  for (int i = threadIdx.x; i < TP * N; i += blockDim.x) {
    int t, pr;
    const int e = dTP.div(i, t), p = p0 + t, pq = dH.div(p, pr);
    cx<T> v = {T(0), T(0)};
    if (p < npen) v = cload(FQ + (size_t)pr + (size_t)pq * S1 + (size_t)e * Se);
    a[t * N + e] = v;
  }
  __syncthreads();
  cx<T> *r = lds_fft<T, S>(a, b, N, N, TP, ax, tw);
  for (int i = threadIdx.x; i < TP * N; i += blockDim.x) {
    int t, pr;
    const int e = dTP.div(i, t), p = p0 + t, pq = dH.div(p, pr);
    if (p < npen) cstore(FQ + (size_t)pr + (size_t)pq * S1 + (size_t)e * Se, r[t * N + e]);
  }
}

// Pencils along K3: forward FFT, influence function (scalar_sum.f:40-121,
// FFTW variant, with its fac12/fac13/fac23 virial masks and the unscaled
// m = 0 term), inverse FFT.  Per-block partials: energy, v11 v22 v33 v12 v13 v23.
template <typename T>
__global__ void __launch_bounds__(256) k_fft_z_conv(const PmeDesc *__restrict__ D) {
  extern __shared__ __align__(16) unsigned char smem[];
  __shared__ double red[8][8];
  const PmeDesc &d = D[blockIdx.y];
  if ((int)blockIdx.x >= d.conv_nblk) return;
  const int H = d.K1 / 2 + 1, N = d.K3, TP = d.tpz;
  const int npen = H * d.K2;
  const size_t Se = (size_t)H * d.K2;
  const int p0 = blockIdx.x * TP;
  double acc[7] = {0, 0, 0, 0, 0, 0, 0};
  const int LD = N + 1;
  cx<T> *FQ = reinterpret_cast<cx<T> *>(d.FQ);
  cx<T> *a = reinterpret_cast<cx<T> *>(smem);
  cx<T> *b = a + TP * LD, *tw = b + TP * LD;
  const FastDiv dTP(TP), dH(H);
  if (p0 < npen) {
    const int nfft1 = d.K1, nfft2 = d.K2, nfft3 = d.K3, ndim1 = H, npt = TP * N;
    int nf1 = nfft1 / 2; if (2 * nf1 < nfft1) nf1 += 1;
    int nf2 = nfft2 / 2; if (2 * nf2 < nfft2) nf2 += 1;
    int nf3 = nfft3 / 2; if (2 * nf3 < nfft3) nf3 += 1;
    const double pi = d.pi_f32, fac = d.fac;
    // 1-based indices as in scalar_sum; false outside the grid and at ind = 0, which is never scaled
    auto point = [&](int i, int &k1, int &k2, int &k3, double (&mh)[3]) -> bool {
      int t, pr;
      const int e = dTP.div(i, t), p = p0 + t, pq = dH.div(p, pr);
      k1 = pr + 1, k2 = pq + 1, k3 = e + 1;
      int m1 = k1 - 1; if (k1 > nf1) m1 = k1 - 1 - nfft1;
      int m2 = k2 - 1; if (k2 > nf2) m2 = k2 - 1 - nfft2;
      int m3 = k3 - 1; if (k3 > nf3) m3 = k3 - 1 - nfft3;
      const double *rc = d.recip;
      mh[0] = rc[0] * m1 + rc[3] * m2 + rc[6] * m3;
      mh[1] = rc[1] * m1 + rc[4] * m2 + rc[7] * m3;
      mh[2] = rc[2] * m1 + rc[5] * m2 + rc[8] * m3;
      return i < npt && p < npen && !(k1 == 1 && k2 == 1 && k3 == 1);
    };
    load_twiddles(tw, d.ax3);
    cx<T> v[CONV_PTS];
#pragma unroll
    for (int c = 0; c < CONV_PTS; ++c) {
      if (c * 256 >= npt) continue;
      int t;
      const int i = c * 256 + threadIdx.x, e = dTP.div(i, t), p = p0 + t;
      v[c] = {T(0), T(0)};
      if (i < npt && p < npen) v[c] = cload(FQ + (size_t)p + (size_t)e * Se);
    }
    // the influence function needs no data: evaluated while the loads are in flight
    double eterm[CONV_PTS], vterm[CONV_PTS];
#pragma unroll
    for (int c = 0; c < CONV_PTS; ++c) {
      if (c * 256 >= npt) continue;
      int k1, k2, k3;
      double mh[3];
      eterm[c] = vterm[c] = 0.0;
      if (!point(c * 256 + threadIdx.x, k1, k2, k3, mh)) continue;
      const double msq = mh[0] * mh[0] + mh[1] * mh[1] + mh[2] * mh[2];
      if (msq > d.rkcut2) continue;
      const double denom = pi * d.volume * gmem(d.bsp1)[k1 - 1] * gmem(d.bsp2)[k2 - 1] * gmem(d.bsp3)[k3 - 1] * msq;
      eterm[c] = exp(-fac * msq) / denom;
      vterm[c] = 2.0 * (fac * msq + 1.0) / msq;
    }
#pragma unroll
    for (int c = 0; c < CONV_PTS; ++c) {
      if (c * 256 >= npt) continue;
      int t;
      const int i = c * 256 + threadIdx.x, e = dTP.div(i, t);
      if (i < npt) a[t * LD + e] = v[c];
    }
    __syncthreads();
    cx<T> *r = lds_fft<T, -1>(a, b, N, LD, TP, d.ax3, tw);
    cx<T> *s = (r == a) ? b : a;
#pragma unroll
    for (int c = 0; c < CONV_PTS; ++c) {
      if (c * 256 >= npt) continue;
      int k1, k2, k3;
      double mh[3];
      if (!point(c * 256 + threadIdx.x, k1, k2, k3, mh)) continue;
      int t;
      const int e = dTP.div(c * 256 + threadIdx.x, t);
      cx<T> &q = r[t * LD + e];
      const double qr = (double)q.x, qi = (double)q.y;
      if (vterm[c] != 0.0) {  // (within the cut-off; vterm is positive there)
        double struc2, f12 = 1.0, f13 = 1.0, f23 = 1.0;
        if (k1 == 1 || (k1 == ndim1 && (nfft1 & 1) == 0)) {
          struc2 = eterm[c] * qr * qr + eterm[c] * qi * qi;
        } else {
          double e2 = 2.0 * eterm[c];
          struc2 = e2 * qr * qr + e2 * qi * qi;
          f12 = (mh[0] * mh[1] < 0.0 && k2 <= ndim1) ? 0.0 : 1.0;
          f13 = (mh[0] * mh[2] < 0.0 && k3 <= ndim1) ? 0.0 : 1.0;
          bool neg = mh[1] * mh[2] < 0.0;
          bool lo2 = k2 <= ndim1, lo3 = k3 <= ndim1;
          f23 = (lo2 == lo3) ? (neg ? 0.0 : 1.0) : (neg ? 1.0 : 0.0);
        }
        double vvir = struc2 * vterm[c];
        acc[0] += struc2;
        acc[1] += struc2 * (vterm[c] * mh[0] * mh[0] - 1.0);
        acc[2] += struc2 * (vterm[c] * mh[1] * mh[1] - 1.0);
        acc[3] += struc2 * (vterm[c] * mh[2] * mh[2] - 1.0);
        acc[4] += vvir * mh[0] * mh[1] * f12;
        acc[5] += vvir * mh[0] * mh[2] * f13;
        acc[6] += vvir * mh[1] * mh[2] * f23;
      }
      q = {T(qr * eterm[c]), T(qi * eterm[c])};
    }
    __syncthreads();
    if (!d.energy_only) {
      cx<T> *o = lds_fft<T, +1>(r, s, N, LD, TP, d.ax3, tw);
      for (int i = threadIdx.x; i < TP * N; i += blockDim.x) {
        int t;
        const int e = dTP.div(i, t), p = p0 + t;
        if (p < npen) cstore(FQ + (size_t)p + (size_t)e * Se, o[t * LD + e]);
      }
    }
  }
  // fixed-order block reduction of the 7 partial sums
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6, nw = blockDim.x >> 6;
#pragma unroll
  for (int k = 0; k < 7; ++k) {
    double v = wave_sum(acc[k]);
    if (lane == 0) red[wid][k] = v;
  }
  __syncthreads();
  if (threadIdx.x < 7) {
    double s = 0.0;
    for (int w = 0; w < nw; ++w) s += red[w][threadIdx.x];
    d.conv_part[(size_t)blockIdx.x * 8 + threadIdx.x] = s;
  }
}

// Half spectrum rows -> real rows (imaginary parts of k1 = 0 and Nyquist ignored).
template <typename T>
__global__ void __launch_bounds__(256) k_fft_x_c2r(const PmeDesc *__restrict__ D) {
  extern __shared__ __align__(16) unsigned char smem[];
  const PmeDesc &d = D[blockIdx.y];
  const int N = d.K1, H = N / 2 + 1, rows = d.K2 * d.K3, TP = d.tpx;
  if ((int)blockIdx.x >= d.gx || d.energy_only || use_planes<T>(d)) return;
  cx<T> *a = reinterpret_cast<cx<T> *>(smem);
  cx<T> *b = a + TP * N;
  cx<T> *tw = b + TP * N;
  const int row0 = blockIdx.x * TP;
  const cx<T> *FQ = reinterpret_cast<const cx<T> *>(d.FQ);
  const FastDiv dN(N), dH(H);
  load_twiddles(tw, d.ax1);
  for (int i = threadIdx.x; i < TP * H; i += blockDim.x) {
    int e;
    const int t = dH.div(i, e), row = row0 + t;
    cx<T> v = {T(0), T(0)};
    if (row < rows) v = cload(FQ + (size_t)row * H + e);
    if (e == 0 || 2 * e == N) v.y = T(0);
    a[t * N + e] = v;
    if (e > 0 && N - e >= H) a[t * N + (N - e)] = {v.x, -v.y};
  }
  __syncthreads();
  cx<T> *r = lds_fft<T, +1>(a, b, N, N, TP, d.ax1, tw);
  T *Qr = reinterpret_cast<T *>(d.Qr);
  for (int i = threadIdx.x; i < TP * N; i += blockDim.x) {
    int e;
    const int t = dN.div(i, e), row = row0 + t;
    if (row < rows) gmem(Qr)[(size_t)row * N + e] = r[t * N + e].x;
  }
}

// ---------------------------------------------------------------- gather

// `order` lanes per atom, 64 / order atoms per wavefront: lane i3 sums the
// z-plane i3 of the atom's order^3 stencil, and the partial f1, f2, f3 are
// summed over the atom's lanes in plane order (fixed order).  Bound by the
// latency of order^2 scattered grid loads a lane: with the order known at
// compile time (ORDER > 0) they are all in flight at once (24,460 atoms, order
// 5: 20 -> 14 us in FP64).  Orders 4 to 6, what simulations use, are written
// out; a launch of other or mixed orders takes the order at run time.
template <typename T, int ORDER>
__global__ void __launch_bounds__(256) k_gather(const PmeDesc *__restrict__ D) {
  __shared__ double red[8][9];
  const PmeDesc &d = D[blockIdx.y];
  if ((int)blockIdx.x >= d.gather_nblk || d.energy_only) return;
  const int order = ORDER > 0 ? ORDER : d.order;
  const int apw = 64 / order;
  const int lane = threadIdx.x & 63;
  const int slot = lane / order, sub = lane - slot * order;
  int a = (blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6)) * apw + slot;
  if (slot >= apw) a = d.natoms;  // lanes past the last whole atom of the wave
  double stc[9] = {0, 0, 0, 0, 0, 0, 0, 0, 0};
  double xp = 0, yp = 0, zp = 0, fr1 = -1, fr2 = -1, fr3 = -1;
  if (a < d.natoms) {
    xp = d.xp[a];
    yp = d.yp[a];
    zp = d.zp[a];
    double x, y, z;
    cartesian(d.co, xp, yp, zp, x, y, z);
    fr1 = frac_coord(x, y, z, d.recip, 0, d.K1);
    fr2 = frac_coord(x, y, z, d.recip, 1, d.K2);
    fr3 = frac_coord(x, y, z, d.recip, 2, d.K3);
  }
  const bool valid =
      a < d.natoms && fr1 >= 0.0 && fr1 <= d.K1 && fr2 >= 0.0 && fr2 <= d.K2 && fr3 >= 0.0 && fr3 <= d.K3;
  double f1 = 0.0, f2 = 0.0, f3 = 0.0;
  int b1 = 0, b2 = 0, b3 = 0;
  if (valid) {
    b1 = (int)fr1;
    b2 = (int)fr2;
    b3 = (int)fr3;
    constexpr int NO = ORDER > 0 ? ORDER : MAX_ORDER;
    T th1[NO], th2[NO], th3[NO], dt1[NO], dt2[NO], dt3[NO];
    const auto Qr = gmem(reinterpret_cast<const T *>(d.Qr));
    const int i3 = sub;
    const int kk = wrapK(b3 - order + i3 + 1, d.K3);
    const unsigned plane = (unsigned)d.K1 * d.K2 * kk;
    if constexpr (ORDER > 0) {
      unsigned ii[NO];
#pragma unroll
      for (int i1 = 0; i1 < NO; ++i1) ii[i1] = plane + wrapK(b1 - NO + i1 + 1, d.K1);
      T g[NO][NO];
#pragma unroll
      for (int i2 = 0; i2 < NO; ++i2) {
        const unsigned row = (unsigned)d.K1 * wrapK(b2 - NO + i2 + 1, d.K2);
#pragma unroll
        for (int i1 = 0; i1 < NO; ++i1) g[i2][i1] = Qr[row + ii[i1]];
      }
      fill_bspline_n<T, ORDER>(T(fr1 - b1), th1, dt1);
      fill_bspline_n<T, ORDER>(T(fr2 - b2), th2, dt2);
      fill_bspline_n<T, ORDER>(T(fr3 - b3), th3, dt3);
      T t3 = th3[0], d3 = dt3[0];  // this lane's plane
#pragma unroll
      for (int k = 1; k < NO; ++k) {
        t3 = i3 == k ? th3[k] : t3;
        d3 = i3 == k ? dt3[k] : d3;
      }
#pragma unroll
      for (int i2 = 0; i2 < NO; ++i2) {
        T s1 = T(0), s23 = T(0);
#pragma unroll
        for (int i1 = 0; i1 < NO; ++i1) {
          s1 += dt1[i1] * g[i2][i1];
          s23 += th1[i1] * g[i2][i1];
        }
        f1 -= (double)(s1 * th2[i2] * t3);
        f2 -= (double)(s23 * dt2[i2] * t3);
        f3 -= (double)(s23 * th2[i2] * d3);
      }
    } else {
      fill_bspline<T>(T(fr1 - b1), order, th1, dt1);
      fill_bspline<T>(T(fr2 - b2), order, th2, dt2);
      fill_bspline<T>(T(fr3 - b3), order, th3, dt3);
      for (int i2 = 0; i2 < order; ++i2) {
        const unsigned row = plane + (unsigned)d.K1 * wrapK(b2 - order + i2 + 1, d.K2);
        T s1 = T(0), s23 = T(0);
        for (int i1 = 0; i1 < order; ++i1) {
          T g = Qr[row + wrapK(b1 - order + i1 + 1, d.K1)];
          s1 += dt1[i1] * g;
          s23 += th1[i1] * g;
        }
        f1 -= (double)(s1 * th2[i2] * th3[i3]);
        f2 -= (double)(s23 * dt2[i2] * th3[i3]);
        f3 -= (double)(s23 * th2[i2] * dt3[i3]);
      }
    }
  }
  {
    // every lane takes part in the shuffles; the atom's lanes are slot*order + k
    const int src0 = (slot < apw ? slot : 0) * order;
    double s1 = 0.0, s2 = 0.0, s3 = 0.0;
    for (int k = 0; k < order; ++k) {
      s1 += __shfl(f1, src0 + k, 64);
      s2 += __shfl(f2, src0 + k, 64);
      s3 += __shfl(f3, src0 + k, 64);
    }
    f1 = s1;
    f2 = s2;
    f3 = s3;
  }
  if (valid && sub == 0) {
    const double q = d.q[a];
    f1 *= d.K1 * q;
    f2 *= d.K2 * q;
    f3 *= d.K3 * q;
    const double *rc = d.recip;
    double fx = rc[0] * f1 + rc[3] * f2 + rc[6] * f3;
    double fy = rc[1] * f1 + rc[4] * f2 + rc[7] * f3;
    double fz = rc[2] * f1 + rc[5] * f2 + rc[8] * f3;
    if (d.accumulate) {
      d.fx[a] += fx;
      d.fy[a] += fy;
      d.fz[a] += fz;
    } else {
      d.fx[a] = fx;
      d.fy[a] = fy;
      d.fz[a] = fz;
    }
    if (d.atomp) {
      int j = d.atomp[a];
      double sx = xp - d.xpcm[j], sy = yp - d.ypcm[j], sz = zp - d.zpcm[j];
      const double *co = d.co;
      double gx = sx * co[0] + sy * co[3] + sz * co[6];
      double gy = sx * co[1] + sy * co[4] + sz * co[7];
      double gz = sx * co[2] + sy * co[5] + sz * co[8];
      stc[0] = -gx * fx; stc[1] = -gy * fx; stc[2] = -gz * fx;
      stc[3] = -gx * fy; stc[4] = -gy * fy; stc[5] = -gz * fy;
      stc[6] = -gx * fz; stc[7] = -gy * fz; stc[8] = -gz * fz;
    }
  }
  const int wid = threadIdx.x >> 6, nw = blockDim.x >> 6;
#pragma unroll
  for (int k = 0; k < 9; ++k) {
    double v = wave_sum(stc[k]);
    if (lane == 0) red[wid][k] = v;
  }
  __syncthreads();
  if (threadIdx.x < 9) {
    double s = 0.0;
    for (int w = 0; w < nw; ++w) s += red[w][threadIdx.x];
    d.gather_part[(size_t)blockIdx.x * 9 + threadIdx.x] = s;
  }
}

__global__ void __launch_bounds__(1024) k_pme_finalize(const PmeDesc *__restrict__ D) {
  pme_finalize(D[blockIdx.y], blockIdx.x);
}

// ---------------------------------------------------------------- launchers

static int tile_pencils(int n, int npen, int elems) {
  // two buffers (pencils n + 1 apart) and the twiddles within 64 KB in FP64
  int tp = std::min(elems / n, (4096 - n) / (2 * (n + 1)));
  if (tp < 1) tp = 1;
  if (tp > npen) tp = npen;
  return tp;
}

// FFT tiling of one system for LDS buffers of lds_elems complex elements
void pme_set_tiles(PmeDesc &d, int lds_elems) {
  const int H = d.K1 / 2 + 1;
  d.tpx = tile_pencils(d.K1, d.K2 * d.K3, lds_elems);
  d.gx = (d.K2 * d.K3 + d.tpx - 1) / d.tpx;
  d.tpy = tile_pencils(d.K2, H * d.K3, lds_elems);
  d.gy = (H * d.K3 + d.tpy - 1) / d.tpy;
  d.tpz = tile_pencils(d.K3, H * d.K2, lds_elems);
  d.conv_nblk = (H * d.K2 + d.tpz - 1) / d.tpz;
  const int apb = 4 * (64 / d.order);     // k_gather: order lanes per atom, 4 waves per block
  d.gather_nblk = (d.natoms + apb - 1) / apb;
}

template <typename T>
void launch_pme(const PmeDesc *d_desc, const PmeDesc *h, int nsys, hipStream_t st, const hipEvent_t *ev, bool finalize,
                bool binned) {
  if (nsys <= 0) return;
  int max_atoms = 1, max_bins = 1, any_tiled = 0, any_atomic = 0, max_gx = 0, max_gy = 0, max_gz = 1, max_gg = 1;
  int max_planes = 0, max_plane = 0;
  int order = 0, max_order = 0;
  size_t max_grid = 1, shx = 0, shy = 0, shz = 0, shp = 0, max_work = 1;
  for (int s = 0; s < nsys; ++s) {
    const PmeDesc &d = h[s];
    max_atoms = std::max(max_atoms, d.natoms);
    if (use_planes<T>(d)) {
      max_planes = std::max(max_planes, d.K3);
      max_plane = std::max(max_plane, d.K1 * d.K2);
      shp = std::max(shp, plane_lds<T>(d));
    } else {
      max_gx = std::max(max_gx, d.gx);
      max_gy = std::max(max_gy, d.gy);
    }
    max_gz = std::max(max_gz, d.conv_nblk);
    max_gg = std::max(max_gg, d.gather_nblk);
    shx = std::max(shx, (2 * (size_t)d.tpx + 1) * d.K1 * sizeof(cx<T>));
    shy = std::max(shy, (2 * (size_t)d.tpy + 1) * d.K2 * sizeof(cx<T>));
    shz = std::max(shz, (2 * (size_t)d.tpz * (d.K3 + 1) + d.K3) * sizeof(cx<T>));
    // one spline order in the whole launch: the kernels written out for it
    order = s == 0 || order == d.order ? d.order : 0;
    max_order = std::max(max_order, d.order);
    if (d.tiled) {
      any_tiled = 1;
      max_bins = std::max(max_bins, d.nb1 * d.nb2 * d.nb3);
    } else {
      any_atomic = 1;
      max_grid = std::max(max_grid, (size_t)d.K1 * d.K2 * d.K3);
      max_work = std::max(max_work, (size_t)d.natoms * d.order);
    }
  }
  dim3 blk(256);
  if (ev) ORAC_HIP(hipEventRecord(ev[0], st));
  if (any_tiled) {
    if (!binned) hipLaunchKernelGGL(k_bin, dim3((max_atoms + 255) / 256, nsys), blk, 0, st, d_desc);
    const dim3 gt(max_bins, nsys), bt(SPREAD_THREADS);
    const size_t sh = spread_lds_bytes<T>(max_order);
    switch (order) {
      case 4: hipLaunchKernelGGL((k_spread_tile<T, 4>), gt, bt, sh, st, d_desc); break;
      case 5: hipLaunchKernelGGL((k_spread_tile<T, 5>), gt, bt, sh, st, d_desc); break;
      case 6: hipLaunchKernelGGL((k_spread_tile<T, 6>), gt, bt, sh, st, d_desc); break;
      default: hipLaunchKernelGGL((k_spread_tile<T, 0>), gt, bt, sh, st, d_desc); break;
    }
  }
  if (any_atomic) {
    unsigned gzero = (unsigned)std::min<size_t>((max_grid + 255) / 256, 4096);
    hipLaunchKernelGGL(k_grid_zero, dim3(gzero, nsys), blk, 0, st, d_desc);
    hipLaunchKernelGGL(k_spread<T>, dim3((unsigned)((max_work + 255) / 256), nsys), blk, 0, st, d_desc);
  }
  if (ev) ORAC_HIP(hipEventRecord(ev[1], st));
  // Threads a plane: up to 64 x 64 two or more workgroups share a compute unit's LDS, and 512 threads
  // let them overlap (12 systems, us with 512 and 1,024: 32^3 37 49, 48^3 68 88, 64^3 115 128 in FP64;
  // one system 1 to 2 us the other way).  Larger planes have the unit to themselves in FP64 (80^3 235
  // 225, 96^3 371 356); in FP32 72^3 to 96^3 still share it in a batch (12 systems of 80^3 156 181), one
  // system not (48 45), and the single one decides.
  const dim3 pl(max_planes, nsys), bp(max_plane <= 64 * 64 ? 512 : 1024);
  if (max_planes) hipLaunchKernelGGL(k_fft_plane_r2c<T>, pl, bp, shp, st, d_desc);
  if (max_gx) {
    hipLaunchKernelGGL(k_fft_x_r2c<T>, dim3(max_gx, nsys), blk, shx, st, d_desc);
    hipLaunchKernelGGL((k_fft_pencil<T, -1>), dim3(max_gy, nsys), blk, shy, st, d_desc);
  }
  hipLaunchKernelGGL(k_fft_z_conv<T>, dim3(max_gz, nsys), blk, shz, st, d_desc);
  if (max_planes) hipLaunchKernelGGL(k_fft_plane_c2r<T>, pl, bp, shp, st, d_desc);
  if (max_gx) {
    hipLaunchKernelGGL((k_fft_pencil<T, +1>), dim3(max_gy, nsys), blk, shy, st, d_desc);
    hipLaunchKernelGGL(k_fft_x_c2r<T>, dim3(max_gx, nsys), blk, shx, st, d_desc);
  }
  if (ev) ORAC_HIP(hipEventRecord(ev[2], st));
  switch (order) {
    case 4: hipLaunchKernelGGL((k_gather<T, 4>), dim3(max_gg, nsys), blk, 0, st, d_desc); break;
    case 5: hipLaunchKernelGGL((k_gather<T, 5>), dim3(max_gg, nsys), blk, 0, st, d_desc); break;
    case 6: hipLaunchKernelGGL((k_gather<T, 6>), dim3(max_gg, nsys), blk, 0, st, d_desc); break;
    default: hipLaunchKernelGGL((k_gather<T, 0>), dim3(max_gg, nsys), blk, 0, st, d_desc); break;
  }
  if (ev) ORAC_HIP(hipEventRecord(ev[3], st));
  if (finalize) hipLaunchKernelGGL(k_pme_finalize, dim3(16, nsys), dim3(1024), 0, st, d_desc);
}

template void launch_pme<double>(const PmeDesc *, const PmeDesc *, int, hipStream_t, const hipEvent_t *, bool, bool);
template void launch_pme<float>(const PmeDesc *, const PmeDesc *, int, hipStream_t, const hipEvent_t *, bool, bool);

}  // namespace orac
