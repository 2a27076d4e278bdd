// ptc_dft.hpp -- complex arithmetic, spectrum access and the small DFTs held in
// registers, shared by the specialised (ptc_fft2.hip) and the run-time length
// (ptc_fft.hip) transforms.
#pragma once

#include "ptc_internal.hpp"

namespace ptc {

namespace f2 {

__device__ __forceinline__ double2 cmul(double2 a, double2 b) {
  return make_double2(a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x);
}
__device__ __forceinline__ double2 cadd(double2 a, double2 b) { return make_double2(a.x + b.x, a.y + b.y); }
__device__ __forceinline__ double2 csub(double2 a, double2 b) { return make_double2(a.x - b.x, a.y - b.y); }
template <bool INV>
__device__ __forceinline__ double2 mul_mi(double2 a) {
  return INV ? make_double2(-a.y, a.x) : make_double2(a.y, -a.x);
}

// spectra are stored as double2 (FP64 form) or float2 (FP32-storage form);
// arithmetic is FP64 either way
__device__ __forceinline__ double2 ld2(const double2 &v) { return v; }
__device__ __forceinline__ double2 ld2(const float2 &v) { return make_double2(v.x, v.y); }
__device__ __forceinline__ void st2(double2 &d, double2 v) { d = v; }
__device__ __forceinline__ void st2(float2 &d, double2 v) { d = make_float2((float)v.x, (float)v.y); }

// Streaming (nontemporal) forms: the access is marked as not to be kept in
// the caches.  A pass over a field larger than the last-level cache reads
// and writes each value once, so keeping it only evicts other data.
typedef double st_d2 __attribute__((ext_vector_type(2)));
typedef float st_f2 __attribute__((ext_vector_type(2)));
__device__ __forceinline__ double2 ld2s(const double2 &v) {
  const st_d2 w = __builtin_nontemporal_load(reinterpret_cast<const st_d2 *>(&v));
  return make_double2(w.x, w.y);
}
__device__ __forceinline__ double2 ld2s(const float2 &v) {
  const st_f2 w = __builtin_nontemporal_load(reinterpret_cast<const st_f2 *>(&v));
  return make_double2(w.x, w.y);
}
__device__ __forceinline__ void st2s(double2 &d, double2 v) {
  st_d2 w = {v.x, v.y};
  __builtin_nontemporal_store(w, reinterpret_cast<st_d2 *>(&d));
}
__device__ __forceinline__ void st2s(float2 &d, double2 v) {
  st_f2 w = {(float)v.x, (float)v.y};
  __builtin_nontemporal_store(w, reinterpret_cast<st_f2 *>(&d));
}
template <bool STREAM, typename S>
__device__ __forceinline__ double2 ld2x(const S &v) {
  if constexpr (STREAM) return ld2s(v);
  else return ld2(v);
}
template <bool STREAM, typename S>
__device__ __forceinline__ void st2x(S &d, double2 v) {
  if constexpr (STREAM) st2s(d, v);
  else st2(d, v);
}

// ---- small DFTs ----
template <int R, bool INV>
struct Dft;
template <bool INV>
struct Dft<2, INV> {
  static __device__ __forceinline__ void run(double2 *v) {
    const double2 a = v[0], b = v[1];
    v[0] = cadd(a, b);
    v[1] = csub(a, b);
  }
};
template <bool INV>
struct Dft<4, INV> {
  static __device__ __forceinline__ void run(double2 *v) {
    const double2 t0 = cadd(v[0], v[2]), t1 = csub(v[0], v[2]);
    const double2 t2 = cadd(v[1], v[3]), t3 = mul_mi<INV>(csub(v[1], v[3]));
    v[0] = cadd(t0, t2);
    v[1] = cadd(t1, t3);
    v[2] = csub(t0, t2);
    v[3] = csub(t1, t3);
  }
};
template <bool INV>
struct Dft<8, INV> {
  static __device__ __forceinline__ void run(double2 *v) {
    constexpr double r2 = 0.70710678118654752440;
    double2 e[4] = {v[0], v[2], v[4], v[6]};
    double2 o[4] = {v[1], v[3], v[5], v[7]};
    Dft<4, INV>::run(e);
    Dft<4, INV>::run(o);
    const double2 o1 = INV ? make_double2(r2 * (o[1].x - o[1].y), r2 * (o[1].x + o[1].y))
                           : make_double2(r2 * (o[1].x + o[1].y), r2 * (o[1].y - o[1].x));
    const double2 o2 = mul_mi<INV>(o[2]);
    const double2 o3 = INV ? make_double2(-r2 * (o[3].x + o[3].y), r2 * (o[3].x - o[3].y))
                           : make_double2(r2 * (o[3].y - o[3].x), -r2 * (o[3].x + o[3].y));
    v[0] = cadd(e[0], o[0]);
    v[4] = csub(e[0], o[0]);
    v[1] = cadd(e[1], o1);
    v[5] = csub(e[1], o1);
    v[2] = cadd(e[2], o2);
    v[6] = csub(e[2], o2);
    v[3] = cadd(e[3], o3);
    v[7] = csub(e[3], o3);
  }
};

template <int R>
struct Trig;
template <>
struct Trig<3> {
  static constexpr double c[3] = {1.0, -0.5, -0.5};
  static constexpr double s[3] = {0.0, 0.86602540378443864676, -0.86602540378443864676};
};
template <>
struct Trig<5> {
  static constexpr double c[5] = {1.0, 0.30901699437494742410, -0.80901699437494742410, -0.80901699437494742410,
                                  0.30901699437494742410};
  static constexpr double s[5] = {0.0, 0.95105651629515357212, 0.58778525229247312917, -0.58778525229247312917,
                                  -0.95105651629515357212};
};
template <>
struct Trig<7> {
  static constexpr double c[7] = {1.0, 0.62348980185873353053, -0.22252093395631440429, -0.90096886790241912624,
                                  -0.90096886790241912624, -0.22252093395631440429, 0.62348980185873353053};
  static constexpr double s[7] = {0.0, 0.78183148246802980871, 0.97492791218182360702, 0.43388373911755812048,
                                  -0.43388373911755812048, -0.97492791218182360702, -0.78183148246802980871};
};

template <int R, bool INV>
struct DftOdd {
  static __device__ __forceinline__ void run(double2 *v) {
    constexpr int H = (R - 1) / 2;
    double2 a[H + 1], b[H + 1];
#pragma unroll
    for (int q = 1; q <= H; ++q) {
      a[q] = cadd(v[q], v[R - q]);
      b[q] = csub(v[q], v[R - q]);
    }
    double2 x0 = v[0];
#pragma unroll
    for (int q = 1; q <= H; ++q) x0 = cadd(x0, a[q]);
    double2 out[R];
    out[0] = x0;
#pragma unroll
    for (int r = 1; r <= H; ++r) {
      double2 A = v[0], B = make_double2(0.0, 0.0);
#pragma unroll
      for (int q = 1; q <= H; ++q) {
        const double cq = Trig<R>::c[(q * r) % R], sq = Trig<R>::s[(q * r) % R];
        A.x += a[q].x * cq;
        A.y += a[q].y * cq;
        B.x += b[q].x * sq;
        B.y += b[q].y * sq;
      }
      if (!INV) {
        out[r] = make_double2(A.x + B.y, A.y - B.x);
        out[R - r] = make_double2(A.x - B.y, A.y + B.x);
      } else {
        out[r] = make_double2(A.x - B.y, A.y + B.x);
        out[R - r] = make_double2(A.x + B.y, A.y - B.x);
      }
    }
#pragma unroll
    for (int r = 0; r < R; ++r) v[r] = out[r];
  }
};
template <bool INV>
struct Dft<3, INV> : DftOdd<3, INV> {};
template <bool INV>
struct Dft<5, INV> : DftOdd<5, INV> {};
template <bool INV>
struct Dft<7, INV> : DftOdd<7, INV> {};
// 9 points as 3 x 3: three 3-point DFTs of the stride-3 subsequences, the
// twiddles w9^(n2 k1), three 3-point DFTs across them; X[k1 + 3 k2]
template <bool INV>
struct Dft<9, INV> {
  static __device__ __forceinline__ void run(double2 *v) {
    // cos and sin of 2 pi k / 9, k = 1, 2, 4
    constexpr double c1 = 0.7660444431189780352024, s1 = 0.6427876096865393263226;
    constexpr double c2 = 0.1736481776669303488517, s2 = 0.9848077530122080593667;
    constexpr double c4 = -0.9396926207859083840541, s4 = 0.3420201433256687330441;
    double2 t[3][3];
#pragma unroll
    for (int n2 = 0; n2 < 3; ++n2) {
      t[n2][0] = v[n2];
      t[n2][1] = v[n2 + 3];
      t[n2][2] = v[n2 + 6];
      Dft<3, INV>::run(t[n2]);
    }
    // w9^k = (cos, -sin) forward, (cos, sin) inverse
    auto tw = [](double2 a, double c, double sn) {
      const double sg = INV ? sn : -sn;
      return make_double2(a.x * c - a.y * sg, a.x * sg + a.y * c);
    };
    t[1][1] = tw(t[1][1], c1, s1);
    t[1][2] = tw(t[1][2], c2, s2);
    t[2][1] = tw(t[2][1], c2, s2);
    t[2][2] = tw(t[2][2], c4, s4);
#pragma unroll
    for (int k1 = 0; k1 < 3; ++k1) {
      double2 u[3] = {t[0][k1], t[1][k1], t[2][k1]};
      Dft<3, INV>::run(u);
      v[k1] = u[0];
      v[k1 + 3] = u[1];
      v[k1 + 6] = u[2];
    }
  }
};

// R = A * B points with A and B coprime (Good-Thomas): A-point DFTs of the
// subsequences n = B n1 + A n2 (mod R) along n1, then B-point DFTs along n2; the
// result of (k1, k2) is X[k] with k = k1 mod A and k = k2 mod B.  No twiddles.
constexpr int inv_mod(int a, int m) {
  for (int q = 1; q < m; ++q)
    if (a * q % m == 1) return q;
  return 0;
}
template <int A, int B, bool INV>
struct DftPfa {
  static __device__ __forceinline__ void run(double2 *v) {
    constexpr int R = A * B, ea = B * inv_mod(B % A, A), eb = A * inv_mod(A % B, B);
    double2 t[B][A];
#pragma unroll
    for (int n2 = 0; n2 < B; ++n2) {
#pragma unroll
      for (int n1 = 0; n1 < A; ++n1) t[n2][n1] = v[(B * n1 + A * n2) % R];
      Dft<A, INV>::run(t[n2]);
    }
#pragma unroll
    for (int k1 = 0; k1 < A; ++k1) {
      double2 u[B];
#pragma unroll
      for (int n2 = 0; n2 < B; ++n2) u[n2] = t[n2][k1];
      Dft<B, INV>::run(u);
#pragma unroll
      for (int k2 = 0; k2 < B; ++k2) v[(ea * k1 + eb * k2) % R] = u[k2];
    }
  }
};
template <bool INV>
struct Dft<6, INV> : DftPfa<2, 3, INV> {};
template <bool INV>
struct Dft<10, INV> : DftPfa<2, 5, INV> {};
template <bool INV>
struct Dft<12, INV> : DftPfa<4, 3, INV> {};
template <bool INV>
struct Dft<14, INV> : DftPfa<2, 7, INV> {};
template <bool INV>
struct Dft<15, INV> : DftPfa<3, 5, INV> {};
// 16 points as 4 x 4: four 4-point DFTs of the stride-4 subsequences, the
// twiddles w16^(n2 k1), four 4-point DFTs across them; X[k1 + 4 k2]
template <bool INV>
struct Dft<16, INV> {
  static __device__ __forceinline__ void run(double2 *v) {
    constexpr double c1 = 0.92387953251128675613, s1 = 0.38268343236508977173, r2 = 0.70710678118654752440;
    double2 t[4][4];
#pragma unroll
    for (int n2 = 0; n2 < 4; ++n2) {
#pragma unroll
      for (int n1 = 0; n1 < 4; ++n1) t[n2][n1] = v[4 * n1 + n2];
      Dft<4, INV>::run(t[n2]);
    }
    auto tw = [](double2 a, double c, double sn) {
      const double sg = INV ? sn : -sn;
      return make_double2(a.x * c - a.y * sg, a.x * sg + a.y * c);
    };
    t[1][1] = tw(t[1][1], c1, s1);
    t[1][2] = tw(t[1][2], r2, r2);
    t[1][3] = tw(t[1][3], s1, c1);
    t[2][1] = tw(t[2][1], r2, r2);
    t[2][2] = mul_mi<INV>(t[2][2]);
    t[2][3] = tw(t[2][3], -r2, r2);
    t[3][1] = tw(t[3][1], s1, c1);
    t[3][2] = tw(t[3][2], -r2, r2);
    t[3][3] = tw(t[3][3], -c1, -s1);
#pragma unroll
    for (int k1 = 0; k1 < 4; ++k1) {
      double2 u[4] = {t[0][k1], t[1][k1], t[2][k1], t[3][k1]};
      Dft<4, INV>::run(u);
#pragma unroll
      for (int k2 = 0; k2 < 4; ++k2) v[k1 + 4 * k2] = u[k2];
    }
  }
};

}  // namespace f2

// Row j and plane k (both 0-based, j within the pass's nj rows) of line q of an
// x pass, in 32 bits: a line is at least 128 bytes, so fewer than 2^31 of them
// fit the device.  (In 64 bits each lane made up to four long divisions before
// its first load: the FP32-storage solve of 1024x256x512 took 3.50 ms, not 3.45.)
// TILED: tiles of tj x tk lines, powers of two, k fastest inside a tile, the tiles k fastest;
// else j fastest.
struct LineAt {
  int j, k;
};
template <bool TILED>
__device__ __forceinline__ LineAt line_at(unsigned q, unsigned nj, unsigned nz, unsigned tj, unsigned tk) {
  if constexpr (TILED) {
    const int sk = __builtin_ctz(tk), st = sk + __builtin_ctz(tj);
    const unsigned tq = q >> st, wq = q & ((1u << st) - 1), ntk = nz >> sk;
    const unsigned t = tq / ntk;
    return LineAt{(int)(t * tj + (wq >> sk)), (int)((tq - t * ntk) * tk + (wq & (tk - 1)))};
  } else {
    const unsigned k = q / nj;
    return LineAt{(int)(q - k * nj), (int)k};
  }
}

// The values of the Poisson source at the pair of points (2m, 2m+1), formed as
// clcPrSrc does (src/m_TScheme.f90:48-77): sudtal times the divergence
// (point_div).  a, b, c: the pairs m-1, m, m+1 of ux; y0, y1: the
// pair of uy in rows j, j+1; z[0..3]: that of uz in planes k-1 .. k+2; dmax: running
// max |divergence|.
__device__ __forceinline__ double2 div_value(const DivSrc &dv, const Geo &geo, double rdyp, double2 a, double2 b,
                                             double2 c, double2 y0, double2 y1, const double2 *z, double &dmax) {
  const double r0 = point_div(geo, rdyp, a.y, b.x, b.y, c.x, y0.x, y1.x, z[0].x, z[1].x, z[2].x, z[3].x);
  const double r1 = point_div(geo, rdyp, b.x, b.y, c.x, c.y, y0.y, y1.y, z[0].y, z[1].y, z[2].y, z[3].y);
  dmax = fmax(dmax, fmax(fabs(r0), fabs(r1)));
  return make_double2(dv.sudtal * r0, dv.sudtal * r1);
}

// One pair of a row, straight into a transform's first stage (rows of which a
// workgroup holds one).  n2 = nx / 2 pairs in a row of rowlen = nx values.
__device__ __forceinline__ double2 div_pair(const DivSrc &dv, const Geo &geo, int n2, int ny, int nz,
                                            long long rowlen, long long jl, long long k, int m, double &dmax) {
  const long long rj = rowlen * (jl + 1 + (long long)(ny + 2) * k);
  const double2 *uxr = reinterpret_cast<const double2 *>(dv.ux + rj);
  const double2 *uyr = reinterpret_cast<const double2 *>(dv.uy + rj);
  const int mm = m > 0 ? m - 1 : n2 - 1, mp = m + 1 < n2 ? m + 1 : 0;
  const double2 a = uxr[mm], b = uxr[m], cc = uxr[mp];
  const double2 y0 = uyr[m], y1 = uyr[m + n2];
  const long long pl = rowlen * (ny + 2);
  double2 z[4];
#pragma unroll
  for (int s = 0; s < 4; ++s) {
    long long kk = k - 1 + s;
    kk = kk < 0 ? kk + nz : (kk >= nz ? kk - nz : kk);
    z[s] = reinterpret_cast<const double2 *>(dv.uz + rj + (kk - k) * pl)[m];
  }
  const double rdyp = geo.met[M_RDYP * geo.nyh + jl + 1];
  return div_value(dv, geo, rdyp, a, b, cc, y0, y1, z, dmax);
}

// The rows of a workgroup's nl lines (q0 ...) into its LDS lines, by columns: a
// thread forms one pair m of K consecutive planes at a time, whose K + 3 planes
// of uz it loads once, and consecutive lanes take consecutive pairs of a row.
// (Formed in the transform's first stage, each pair loaded all nine of its
// values, four to sixteen lanes to a row.)  Lines come in groups of K planes,
// nzp = nz rounded up to whole groups of them, nlines = rows times nzp: the
// lines of planes past nz are zero and never stored.  slot(l, m): element m of
// the workgroup's line l.
template <int K, class Slot>
__device__ __forceinline__ void div_columns(const DivSrc &dv, const Geo &geo, int n2, int ny, int nz, int nzp,
                                            long long rowlen, int j0, unsigned nlines, int tj, int tk, unsigned q0,
                                            int nl, int nthr, const Slot &slot, double &dmax) {
  const long long pl = rowlen * (ny + 2);
  const int ncol = n2 * (nl / K);
  for (int c = threadIdx.x; c < ncol; c += nthr) {
    const int grp = (unsigned)c / (unsigned)n2, m = c - grp * n2;
    const unsigned q = q0 + grp * K;
    const bool on = q < nlines;
    const LineAt at = line_at<true>(on ? q : 0, 1, nzp, tj, tk);
    const int j = j0 + at.j + 1, k = at.k;
    const long long rj = rowlen * (j + (long long)(ny + 2) * k);
    const int mm = m > 0 ? m - 1 : n2 - 1, mp = m + 1 < n2 ? m + 1 : 0;
    double2 z[K + 3], a[K], b[K], cc[K], y0[K], y1[K];
#pragma unroll
    for (int s = 0; s < K + 3; ++s) {
      int kk = min(k - 1 + s, nz + 1);
      kk = kk < 0 ? kk + nz : (kk >= nz ? kk - nz : kk);
      z[s] = reinterpret_cast<const double2 *>(dv.uz + rj + (kk - k) * pl)[m];
    }
#pragma unroll
    for (int i = 0; i < K; ++i) {
      const long long o = rj + (min(k + i, nz - 1) - k) * pl;
      const double2 *uxr = reinterpret_cast<const double2 *>(dv.ux + o);
      const double2 *uyr = reinterpret_cast<const double2 *>(dv.uy + o);
      a[i] = uxr[mm];
      b[i] = uxr[m];
      cc[i] = uxr[mp];
      y0[i] = uyr[m];
      y1[i] = uyr[m + n2];
    }
    const double rdyp = geo.met[M_RDYP * geo.nyh + j];
#pragma unroll
    for (int i = 0; i < K; ++i) {
      double d = 0.0;
      const double2 v = div_value(dv, geo, rdyp, a[i], b[i], cc[i], y0[i], y1[i], z + i, d);
      const bool live = on && k + i < nz;
      if (live) dmax = fmax(dmax, d);
      slot(grp * K + i, m) = live ? v : make_double2(0.0, 0.0);
    }
  }
}

// the maximum of v over a workgroup by a fixed-order tree in red (one value
// per thread), after a barrier that ends earlier uses of that memory
__device__ __forceinline__ double block_max_tree(double v, double *red) {
  const int t = threadIdx.x;
  __syncthreads();
  red[t] = v;
  __syncthreads();
  for (int n = blockDim.x; n > 1;) {
    const int h = (n + 1) / 2;
    if (t < n - h) red[t] = fmax(red[t], red[t + h]);
    __syncthreads();
    n = h;
  }
  return red[0];
}

// line tiles of the neighbour-reading x passes: the largest of 8, 4, 2, 1 rows
// dividing nj, of 16, 8, 4, 2, 1 planes dividing nz
inline void line_tile(int nj, int nz, int *tj, int *tk) {
  *tj = 8;
  *tk = 16;
  while (nj % *tj) *tj /= 2;
  while (nz % *tk) *tk /= 2;
}

}  // namespace ptc
