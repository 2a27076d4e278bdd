// ptc_spectra.hip -- the energy spectra of clcStat on the device
// (src/m_FlowCase.f90:430-805; the helpers clcEnergySpectraX/Z, clcLTS_*,
// clcCospectraX/Z, clcEnergySpectra2D, clcCosSpectra2D at :954-1375).
//
// The reference transforms each field with R2HC along x (and, separately,
// along z, and for the 2-D spectra along x then z) and sums products of the
// half-complex values over the other direction.  Here each field goes once
// through the Poisson solver's forward x and z passes, in FP64, giving the
// 2-D spectrum F(kx, kz) of every row (kx = 0..nx/2, kz = 0..nz-1), and every
// quantity is read off F:
//   - x spectra: the z sum of Xa(kx, z) conj Xb(kx, z) over z equals
//     (1/nz) sum over kz of Fa conj Fb (Parseval along z);
//   - z spectra: the x sum of Za(x, kz) conj Zb(x, kz) equals (1/nx) times the
//     sum over kx = 0..nx/2 of P(kx, kz) plus the sum over kx = 1..nx/2-1 of
//     conj P(kx, -kz), P = Fa conj Fb (Parseval along x, F(-kx, kz) =
//     conj F(kx, -kz) for real fields);
//   - 2-D spectra: the R2HC along z of the real and imaginary parts of the x
//     transform are (F(kx, kz) + conj F(kx, -kz)) / 2 and
//     (F(kx, kz) - conj F(kx, -kz)) / 2i.
// The linear-coherence spectra are the real and imaginary parts of the same
// sums with b the reference row.  The reference's uCRF shift of ux only moves
// F(0, 0) by nx nz uCRF, which the partial sums add.  The cell-centre ux
// (the 4-point interpolation ic1 ux(i-1) + ic2 ux(i) + ic3 ux(i+1) + ic4 ux(i+2)
// + uCRF) is not transformed separately: its spectrum is H(kx) F_ux(kx, kz)
// with H = ic1 w + ic2 + ic3 conj(w) + ic4 conj(w)^2, w = exp(-2 pi i kx / nx),
// plus the same shift.  Nor is the cell-centre uy, the mean of two face rows: its
// spectrum is the mean of theirs (uy's row ny+1 is transformed by itself).
#include "ptc_internal.hpp"

#include <algorithm>
#include <cmath>
#include <cstring>
#include <vector>

namespace ptc {

namespace {

// Largest partial-sum workgroup.  With 320 threads the 2^k + 1 kx of a power of two
// fit fewer kx per thread (257 one, 513 two), but two loads per thread in flight
// serve better than one: a sample (us, 256 / 320 threads) of 512x128x256 599 / 650,
// 512x96x192 384 / 409, 540x96x128 312 / 331, 600x64x128 251-256 / 259, 1024x128x192
// 858 / 868; the other way 512x32x64 136 / 130, 1024x64x128 343 / 334; 250 to 400 and
// 768 to 2048 points otherwise within 1 %, 384 and 512 threads as 320.
constexpr int kSpecThreads = 256;
constexpr size_t kSpecStage = size_t(2) << 20;  // bytes of a pinned half
constexpr int kSpecRows = 16;      // kz rows per partial-sum workgroup

// ---- row ny+1 of a field as row 1 of a field of one row
__global__ void __launch_bounds__(256) k_spec_top(Geo g, const double *__restrict__ u, double *__restrict__ out) {
  const int i = blockIdx.x * 256 + threadIdx.x, k = blockIdx.y;
  if (i < g.nx) out[(long long)g.nx * (3LL * k + 1) + i] = u[(long long)g.nx * (g.ny + 1) + g.plane * k + i];
}

__device__ inline double2 cmul(double2 a, double2 b) { return make_double2(a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x); }

// The products of one field's spectrum a, summed over kz and over kx.  kEnergy:
// |a|^2.  kSet (a = ux): |a|^2; a conj a(reference row jr1 below row jsplit, jr2
// from it on), complex; a conj c and (hx a) conj c, real parts, with c the
// cell-centre uy from the rows j and j+1 of v (vtop for row ny+1).  sa is added to
// Re F(0, 0) of a (after the multiplication by hx).
enum { kEnergy = 0, kSet = 1 };
struct SpecIn {
  const double2 *a, *v, *vtop, *hx;
  double sa;
  int jr1, jr2, jsplit;
};
// products formed as sums over kz per kx (px), and sums over all kx and over
// 0 < kx < h per kz (pz: two per product)
constexpr int spec_products(int mode) { return mode == kEnergy ? 1 : 5; }

// Partial sums of one row j, kSpecRows kz rows and a segment of kx (grid: x = kz
// chunk, y = j, z = segment of blockDim * NS kx):
//   px[((q * ny + j) * nch + chunk) * (h+1) + kx]       = sum over the chunk's kz
//   pz[(((2 q + inner) * ny + j) * nz + kz) * nseg + seg] = sum over the segment's
//                                            kx, all or only those in 1..h-1
// of product q.  Thread t owns kx = seg start + t + blockDim s, s < NS.  All
// products of a field come from one read of its spectrum, and the sums over kx of
// a batch of rows are exchanged together (wave_sums): one product per launch with
// six exchanges per value read the ux and uy spectra seven times and took 78 us
// a product at 512x128x256, where one read takes about 27.
constexpr int kSpecMaxNs = 4;
template <int NS, int MODE>
constexpr int spec_batch() {
  return MODE == kEnergy ? (NS == 1 ? 8 : NS <= 2 ? 4 : 2) : (NS == 1 ? 4 : NS <= 2 ? 2 : 1);
}

template <int NS, int MODE>
__global__ void __launch_bounds__(kSpecThreads) k_spec_sums(SpecIn S, int ny, int nz, int h, int pitch,
                                                            double *__restrict__ px, double *__restrict__ pz) {
  constexpr int NW = kSpecThreads / 64, NQ = spec_products(MODE), RB = spec_batch<NS, MODE>(), NV = 2 * NQ;
  __shared__ double red[kSpecRows][NW][NV];
  const int j = blockIdx.y, ch = blockIdx.x, nch = gridDim.x;
  const int t = threadIdx.x, nt = blockDim.x, lane = t & 63, w = t >> 6, nw = nt >> 6;
  const int k0 = ch * kSpecRows, k1 = min(nz, k0 + kSpecRows);
  const int kx0 = (int)blockIdx.z * nt * NS + t;
  const int jr = j < S.jsplit ? S.jr1 : S.jr2;
  double sx[NS][NQ];
  double2 hs[NS];
#pragma unroll
  for (int s = 0; s < NS; ++s) {
#pragma unroll
    for (int q = 0; q < NQ; ++q) sx[s][q] = 0.0;
    if (MODE == kSet) hs[s] = S.hx[min(kx0 + nt * s, h)];
  }
  struct Row {
    double2 a, b, v0, v1;
  };
  auto load = [&](int kz, int kx) {
    Row r{};
    const long long base = (long long)kz * ny;
    r.a = S.a[(base + j) * pitch + kx];
    if constexpr (MODE == kSet) {
      r.b = S.a[(base + jr) * pitch + kx];
      r.v0 = S.v[(base + j) * pitch + kx];
      r.v1 = j + 1 < ny ? S.v[(base + j + 1) * pitch + kx] : S.vtop[(long long)kz * pitch + kx];
    }
    return r;
  };
  // the products of one mode into the sums over kz and the row's values
  auto add = [&](const Row &r, int kz, int kx, double2 hx, double (&s)[NQ], double *v) {
    double2 a = r.a;
    const bool origin = kz == 0 && kx == 0;
    double pr[NQ];
    if constexpr (MODE == kSet) {
      double2 b = r.b, ha = cmul(a, hx);
      if (origin) {
        b.x += S.sa;
        ha.x += S.sa;
      }
      const double2 c = make_double2(0.5 * (r.v0.x + r.v1.x), 0.5 * (r.v0.y + r.v1.y));
      if (origin) a.x += S.sa;
      pr[1] = a.x * b.x + a.y * b.y;
      pr[2] = a.y * b.x - a.x * b.y;
      pr[3] = a.x * c.x + a.y * c.y;
      pr[4] = ha.x * c.x + ha.y * c.y;
    }
    pr[0] = a.x * a.x + a.y * a.y;
    const bool inner = kx > 0 && kx < h;
#pragma unroll
    for (int q = 0; q < NQ; ++q) {
      s[q] += pr[q];
      v[2 * q] += pr[q];
      v[2 * q + 1] += inner ? pr[q] : 0.0;
    }
  };
  for (int kb = k0; kb < k1; kb += RB) {
    Row row[RB][NS];
#pragma unroll
    for (int r = 0; r < RB; ++r)
#pragma unroll
      for (int s = 0; s < NS; ++s) row[r][s] = load(min(kb + r, k1 - 1), min(kx0 + nt * s, h));
    double q[RB * NV];
#pragma unroll
    for (int e = 0; e < RB * NV; ++e) q[e] = 0.0;
#pragma unroll
    for (int r = 0; r < RB; ++r)
#pragma unroll
      for (int s = 0; s < NS; ++s)
        if (kb + r < k1 && kx0 + nt * s <= h) add(row[r][s], kb + r, kx0 + nt * s, hs[s], sx[s], q + r * NV);
    int idx;
    wave_sums<RB * NV>(q, lane, &idx);
    if (idx >= 0 && kb + idx / NV < k1) red[kb - k0 + idx / NV][w][idx % NV] = q[0];
  }
#pragma unroll
  for (int q = 0; q < NQ; ++q) {
    double *ox = px + (((long long)q * ny + j) * nch + ch) * (h + 1);
#pragma unroll
    for (int s = 0; s < NS; ++s)
      if (kx0 + nt * s <= h) ox[kx0 + nt * s] = sx[s][q];
  }
  __syncthreads();
  for (int e = t; e < (k1 - k0) * NV; e += nt) {
    const int r = e / NV, v = e - r * NV;
    double sum = 0.0;
    for (int qw = 0; qw < nw; ++qw) sum += red[r][qw][v];
    pz[(((long long)v * ny + j) * nz + k0 + r) * gridDim.z + blockIdx.z] = sum;
  }
}

// Adds one sample to the 1-D accumulators (grid: x = product, y = row j, z = 0 for
// the sums over kz, 1 for those over kx).
// Products of kEnergy: an energy into quantity m (weight 2 inside, 1 at kx = 0,
// nx/2).  Products of kSet: the energy (1), the linear coherence's real (7) and
// imaginary part (8, zero at the edge wavenumbers), no weight, and two
// co-spectra (5, 6), weighted.  ex(kx, j, m) and ez(kz, j, m) are column-major as
// EnergySpecX/Z; m is 1-based.
__global__ void __launch_bounds__(256) k_spec_fin(const double *__restrict__ px, const double *__restrict__ pz,
                                                  int nch, int nseg, int ny, int nx, int nz, int mode, int m,
                                                  double *__restrict__ ex, double *__restrict__ ez) {
  const int j = blockIdx.y, q = blockIdx.x, h = nx / 2, nzh = nz / 2;
  const bool imag = mode == kSet && q == 2, coh = mode == kSet && (q == 1 || q == 2);
  constexpr int set_m[5] = {1, 7, 8, 5, 6};
  const int m0 = (mode == kSet ? set_m[q] : m) - 1;
  // normEgy of the x and z helpers (:962, :1048)
  const double normx = 1.0 / ((double)nx * (double)nx * (double)nz);
  const double normz = 1.0 / ((double)nx * (double)nz * (double)nz);
  const double *pq = px + ((long long)q * ny + j) * nch * (h + 1);
  for (int kx = threadIdx.x; blockIdx.z == 0 && kx <= h; kx += blockDim.x) {
    const bool edge = kx == 0 || kx == h;
    if (imag && edge) continue;
    double sr = 0.0;
    for (int c = 0; c < nch; ++c) sr += pq[(long long)c * (h + 1) + kx];
    sr = sr / (double)nz;
    ex[kx + (long long)(h + 1) * (j + (long long)ny * m0)] += sr * (coh || edge ? 1.0 : 2.0) * normx;
  }
  auto zsum = [&](int in, int kz) {
    const double *pq2 = pz + (((long long)(2 * q + in) * ny + j) * nz + kz) * nseg;
    double s = 0.0;
    for (int g = 0; g < nseg; ++g) s += pq2[g];
    return s;
  };
  for (int kz = threadIdx.x; blockIdx.z == 1 && kz <= nzh; kz += blockDim.x) {
    const bool edge = kz == 0 || kz == nzh;
    if (imag && edge) continue;
    const int km = kz == 0 ? 0 : nz - kz;
    const double v = (imag ? zsum(0, kz) - zsum(1, km) : zsum(0, kz) + zsum(1, km)) / (double)nx;
    ez[kz + (long long)(nzh + 1) * (j + (long long)ny * m0)] += v * (coh || edge ? 1.0 : 2.0) * normz;
  }
}

// The value at half-complex position (p, q) of the R2HC along x then z of
// spectral row `row` (0-based): p <= h is the real part of the x transform at
// kx = p, p > h its imaginary part at kx = nx - p; q likewise along z.
// hx (may be null) multiplies F first and shift is then added to Re F(0, 0).
// cell: the mean of rows row and row+1 (top past row ny-1).
__device__ inline double hc2d_value(const double2 *__restrict__ F, const double2 *__restrict__ top, bool cell,
                                    const double2 *__restrict__ hx, double shift, int ny, int nx, int nz, int pitch,
                                    int row, int p, int q) {
  const int h = nx / 2, nzh = nz / 2;
  const int kx = p <= h ? p : nx - p, kz = q <= nzh ? q : nz - q, km = kz == 0 ? 0 : nz - kz;
  auto at = [&](int k) {
    double2 f = F[((long long)k * ny + row) * pitch + kx];
    if (cell) {
      const double2 g = row + 1 < ny ? F[((long long)k * ny + row + 1) * pitch + kx] : top[(long long)k * pitch + kx];
      f = make_double2(0.5 * (f.x + g.x), 0.5 * (f.y + g.y));
    }
    return hx ? cmul(f, hx[kx]) : f;
  };
  double2 f1 = at(kz), f2 = at(km);
  if (kx == 0 && kz == 0) {
    f1.x += shift;
    f2.x += shift;
  }
  if (p <= h) return q <= nzh ? 0.5 * (f1.x + f2.x) : 0.5 * (f1.y - f2.y);
  return q <= nzh ? 0.5 * (f1.y + f2.y) : 0.5 * (f2.x - f1.x);
}

// Adds one sample to the 2-D accumulator of quantity m (grid: x = p / 64,
// y = chosen row, z = q).  b is a's row, or (top not null) the cell-centre uy's.
// mirror: 0 none (half channel), 1 the row ny+1-jct, 2 the face row ny+2-jct (uy);
// rcoe weighs the mirror's product.
__global__ void __launch_bounds__(64) k_spec_2d(const double2 *__restrict__ a, const double2 *__restrict__ b,
                                                const double2 *__restrict__ top, const double2 *__restrict__ ha,
                                                double sa, int ny, int nx, int nz, int pitch,
                                                const int *__restrict__ iy, int ny2d, int mirror, double rcoe,
                                                double norm, double *__restrict__ out) {
  const int p = blockIdx.x * 64 + threadIdx.x, jc = blockIdx.y, q = blockIdx.z;
  if (p >= nx) return;
  const int jct = iy[jc];
  const bool cell = top != nullptr;
  double v = hc2d_value(a, nullptr, false, ha, sa, ny, nx, nz, pitch, jct - 1, p, q) *
             hc2d_value(b, top, cell, nullptr, 0.0, ny, nx, nz, pitch, jct - 1, p, q);
  if (mirror) {
    const int jcs = (mirror == 2 ? ny + 2 : ny + 1) - jct;
    v += rcoe * (hc2d_value(a, nullptr, false, ha, sa, ny, nx, nz, pitch, jcs - 1, p, q) *
                 hc2d_value(b, top, cell, nullptr, 0.0, ny, nx, nz, pitch, jcs - 1, p, q));
  }
  out[p + (long long)nx * (jc + (long long)ny2d * q)] += norm * v;
}

// launch shape of the partial sums: kx per thread, threads, segments of kx
void sums_shape(int h, int *ns, int *nt, int *nseg) {
  *ns = std::min(kSpecMaxNs, (h + kSpecThreads) / kSpecThreads);
  *nt = std::min(kSpecThreads, ((h + *ns) / *ns + 63) / 64 * 64);
  *nseg = (h + *nt * *ns) / (*nt * *ns);
}

template <int NS>
void sums_launch(ptc_ctx *c, const SpecIn &S, int mode, int nt, int nseg) {
  SpectraState &st = c->spec;
  const dim3 grid((unsigned)st.nch, (unsigned)c->ny, (unsigned)nseg), blk((unsigned)nt);
  if (mode == kSet)
    hipLaunchKernelGGL((k_spec_sums<NS, kSet>), grid, blk, 0, c->stream, S, c->ny, c->nz, c->nx / 2, st.pitch, st.d_px,
                       st.d_pz);
  else
    hipLaunchKernelGGL((k_spec_sums<NS, kEnergy>), grid, blk, 0, c->stream, S, c->ny, c->nz, c->nx / 2, st.pitch,
                       st.d_px, st.d_pz);
}

// the 1-D quantities of one field: kEnergy into quantity m (1-based as the
// reference's), kSet into 1, 5, 6, 7, 8
int spec_1d(ptc_ctx *c, const SpecIn &in, int mode, int m) {
  SpectraState &S = c->spec;
  int ns, nt, nseg;
  sums_shape(c->nx / 2, &ns, &nt, &nseg);
  switch (ns) {
    case 1: sums_launch<1>(c, in, mode, nt, nseg); break;
    case 2: sums_launch<2>(c, in, mode, nt, nseg); break;
    case 3: sums_launch<3>(c, in, mode, nt, nseg); break;
    default: sums_launch<4>(c, in, mode, nt, nseg); break;
  }
  PTC_HIP(hipGetLastError());
  hipLaunchKernelGGL(k_spec_fin, dim3((unsigned)spec_products(mode), (unsigned)c->ny, 2), dim3(256), 0, c->stream, S.d_px,
                     S.d_pz, S.nch, nseg, c->ny, c->nx, c->nz, mode, m, S.d_x, S.d_z);
  PTC_HIP(hipGetLastError());
  return PTC_OK;
}

int spec_2d(ptc_ctx *c, const double2 *a, const double2 *b, int m, int mirror, double rcoe,
            const double2 *top = nullptr, const double2 *ha = nullptr, double sa = 0.0) {
  SpectraState &S = c->spec;
  const int nx = c->nx, nz = c->nz;
  // normEgy of clcEnergySpectra2D / clcCosSpectra2D (:1253-1255)
  double norm = 1.0 / ((double)nx * (double)nz);
  norm = norm * norm;
  if (c->prm.flow_type == 1) norm = norm * 0.5;
  double *out = S.d_2d + (long long)nx * S.ny2d * nz * (m - 1);
  const dim3 grid((unsigned)((nx + 63) / 64), (unsigned)S.ny2d, (unsigned)nz);
  hipLaunchKernelGGL(k_spec_2d, grid, dim3(64), 0, c->stream, a, b, top, ha, sa, c->ny, nx, nz, S.pitch, S.d_iy2d,
                     S.ny2d, c->prm.flow_type == 1 ? mirror : 0, rcoe, norm, out);
  PTC_HIP(hipGetLastError());
  return PTC_OK;
}

// the FP64 2-D spectrum of rows 1..ny of a field
int forward(ptc_ctx *c, const double *src, double2 *spec) {
  PTC_TRY(launch_fft_x_fwd(c, src, spec, true));
  return launch_fft_z(c, spec, false, true);
}

// the 2-D spectrum of uy's row ny+1, through a context of one row
int forward_top(ptc_ctx *c, const double *uy) {
  SpectraState &S = c->spec;
  hipLaunchKernelGGL(k_spec_top, dim3((unsigned)((c->nx + 255) / 256), (unsigned)c->nz), dim3(256), 0, c->stream, c->geo,
                     uy, S.d_toprow);
  PTC_HIP(hipGetLastError());
  ptc_ctx one(*c);  // the launchers read its sizes and plan only
  one.ny = 1;
  return forward(&one, S.d_toprow, S.d_top);
}

template <typename T>
int alloc(T **p, size_t n) {
  PTC_HIP(hipMalloc((void **)p, sizeof(T) * n));
  return PTC_OK;
}

template <typename T>
void release(T *&p) {
  if (p) (void)hipFree(p);
  p = nullptr;
}

size_t n1d_x(const ptc_ctx *c) { return (size_t)(c->nx / 2 + 1) * c->ny * c->spec.ne1; }
size_t n1d_z(const ptc_ctx *c) { return (size_t)(c->nz / 2 + 1) * c->ny * c->spec.ne1; }
size_t n2d(const ptc_ctx *c) { return (size_t)c->nx * c->spec.ny2d * c->nz * c->spec.ne2; }

// work buffers sized by the current Poisson plan's spectral pitch
int ensure_work(ptc_ctx *c) {
  SpectraState &S = c->spec;
  // (the last of them to be allocated: after a failed allocation the next call starts again)
  if (S.d_hx && S.pitch == c->pp.pitch) return PTC_OK;
  release(S.d_fa);
  release(S.d_fb);
  release(S.d_toprow);
  release(S.d_top);
  release(S.d_px);
  release(S.d_pz);
  release(S.d_hx);
  S.pitch = c->pp.pitch;
  S.nch = (c->nz + kSpecRows - 1) / kSpecRows;
  const size_t nspec = (size_t)S.pitch * c->ny * c->nz;
  PTC_TRY(alloc(&S.d_fa, nspec));
  PTC_TRY(alloc(&S.d_fb, nspec));
  PTC_TRY(alloc(&S.d_toprow, (size_t)3 * c->nx * c->nz));
  PTC_TRY(alloc(&S.d_top, (size_t)S.pitch * c->nz));
  PTC_TRY(alloc(&S.d_px, (size_t)spec_products(kSet) * c->ny * S.nch * (c->nx / 2 + 1)));
  int ns, nt, nseg;
  sums_shape(c->nx / 2, &ns, &nt, &nseg);
  PTC_TRY(alloc(&S.d_pz, (size_t)2 * spec_products(kSet) * c->ny * c->nz * nseg));
  // the symbol of the cell-centre interpolation of ux, kx = 0..nx/2
  const int h = c->nx / 2;
  const double ic[4] = {c->geo.ic1, c->geo.ic2, c->geo.ic3, c->geo.ic4};
  std::vector<double2> hx(h + 1);
  for (int kx = 0; kx <= h; ++kx) {
    const double th = 2.0 * M_PI * (double)kx / (double)c->nx;
    const double cs = std::cos(th), sn = std::sin(th), c2 = std::cos(2.0 * th), s2 = std::sin(2.0 * th);
    // ic1 e^{-i th} + ic2 + ic3 e^{i th} + ic4 e^{2 i th}
    hx[kx] = make_double2(ic[0] * cs + ic[1] + ic[2] * cs + ic[3] * c2, -ic[0] * sn + ic[2] * sn + ic[3] * s2);
  }
  PTC_TRY(alloc(&S.d_hx, hx.size()));
  PTC_HIP(hipMemcpy(S.d_hx, hx.data(), sizeof(double2) * hx.size(), hipMemcpyHostToDevice));
  return PTC_OK;
}

}  // namespace

void spectra_free(ptc_ctx *c) {
  SpectraState &S = c->spec;
  release(S.d_x);
  release(S.d_z);
  release(S.d_2d);
  release(S.d_iy2d);
  release(S.d_fa);
  release(S.d_fb);
  release(S.d_toprow);
  release(S.d_top);
  release(S.d_px);
  release(S.d_pz);
  release(S.d_hx);
  for (int q = 0; q < 2; ++q) {
    if (S.h_stage[q]) (void)hipHostFree(S.h_stage[q]);
    if (S.stage_ev[q]) (void)hipEventDestroy(S.stage_ev[q]);
  }
  S = SpectraState{};
}

// InitStatVar's spectra part (src/m_FlowCase.f90:140-251)
int spectra_init(ptc_ctx *c, int clc1d, int jlcs, int clc2d, int ny2d, const int *iy2d) {
  PTC_HIP(hipStreamSynchronize(c->stream));
  spectra_free(c);
  SpectraState &S = c->spec;
  const bool ch = c->prm.flow_type == 1;
  if (ny2d < 1) clc2d = 0;  // :209
  PTC_CHECK(!clc1d || (jlcs >= 1 && jlcs <= c->ny), PTC_E_ARG, "jForLCS outside 1..nyc");
  if (clc2d) {
    PTC_CHECK(iy2d != nullptr, PTC_E_ARG, "null iySpec2D");
    for (int q = 0; q < ny2d; ++q) {
      // :220-232
      if (ch) PTC_CHECK(iy2d[q] >= 2 && iy2d[q] <= c->ny / 2, PTC_E_ARG, "iySpec2D WRONG 1");
      else PTC_CHECK(iy2d[q] >= 2 && iy2d[q] <= c->ny, PTC_E_ARG, "iySpec2D WRONG 2");
    }
  }
  S.on1d = clc1d != 0;
  S.on2d = clc2d != 0;
  S.jlcs = jlcs;
  S.ne1 = c->prm.scalar ? 9 : 8;
  S.ne2 = c->prm.scalar ? 6 : 5;
  S.ny2d = S.on2d ? ny2d : 0;
  if (S.on1d) {
    PTC_TRY(alloc(&S.d_x, n1d_x(c)));
    PTC_TRY(alloc(&S.d_z, n1d_z(c)));
    PTC_TRY(fill_device(c, S.d_x, (long long)n1d_x(c), 0.0));
    PTC_TRY(fill_device(c, S.d_z, (long long)n1d_z(c), 0.0));
  }
  if (S.on2d) {
    S.iy2d.assign(iy2d, iy2d + ny2d);
    PTC_TRY(alloc(&S.d_iy2d, (size_t)ny2d));
    PTC_HIP(hipMemcpy(S.d_iy2d, S.iy2d.data(), sizeof(int) * ny2d, hipMemcpyHostToDevice));
    PTC_TRY(alloc(&S.d_2d, n2d(c)));
    PTC_TRY(fill_device(c, S.d_2d, (long long)n2d(c), 0.0));
  }
  if (S.on1d || S.on2d)
    for (int q = 0; q < 2; ++q) {
      PTC_HIP(hipHostMalloc(reinterpret_cast<void **>(&S.h_stage[q]), kSpecStage, hipHostMallocDefault));
      PTC_HIP(hipEventCreateWithFlags(&S.stage_ev[q], hipEventDisableTiming));
    }
  S.ready = true;
  return PTC_OK;
}

// One sample (src/m_FlowCase.f90:430-805), in the order that keeps two
// spectra live: uy in fb throughout, each other field in fa.
int spectra_sample(ptc_ctx *c, const double *ux, const double *uy, const double *uz, const double *p,
                   const double *sc) {
  SpectraState &S = c->spec;
  PTC_CHECK(S.ready, PTC_E_STATE, "spectra: call ptc_init_spectra first");
  PTC_CHECK(c->pp.ready, PTC_E_STATE, "spectra: the forward transforms need InitPoissonSolver");
  if (!S.on1d && !S.on2d) {
    ++S.nspectime;
    return PTC_OK;
  }
  PTC_TRY(ensure_work(c));
  const int ny = c->ny;
  const double crf = (double)c->nx * (double)c->nz * c->prm.ucrf;  // ux + uCRF moves F(0, 0) only
  // uy -> fb: energy (2); 2-D (2, the face mirror)
  SpecIn P{};
  PTC_TRY(forward(c, uy, S.d_fb));
  PTC_TRY(forward_top(c, uy));
  P.a = S.d_fb;
  if (S.on1d) PTC_TRY(spec_1d(c, P, kEnergy, 2));
  if (S.on2d) PTC_TRY(spec_2d(c, S.d_fb, S.d_fb, 2, 2, 1.0));
  // ux -> fa: energy (1), linear coherence (7, 8), co-spectra with the
  // cell-centre uy of ux + uCRF (5) and of the cell-centre ux (6, H(kx) fa);
  // 2-D: ux (1) and the cell-centre co-spectrum (5, IsSymmetry = .false.: rCoe = -1)
  PTC_TRY(forward(c, ux, S.d_fa));
  if (S.on1d) {
    // :473-489: rows 1..nyc/2 against jForLCS, a channel's upper rows against nyc+1-jForLCS
    const bool ch = c->prm.flow_type == 1;
    P = SpecIn{S.d_fa, S.d_fb, S.d_top, S.d_hx, crf, S.jlcs - 1, ch ? ny - S.jlcs : S.jlcs - 1, ch ? ny / 2 : ny};
    PTC_TRY(spec_1d(c, P, kSet, 0));
  }
  if (S.on2d) {
    PTC_TRY(spec_2d(c, S.d_fa, S.d_fa, 1, 1, 1.0));
    PTC_TRY(spec_2d(c, S.d_fa, S.d_fb, 5, 1, -1.0, S.d_top, S.d_hx, crf));
  }
  // uz, p, scalar
  const double *rest[3] = {uz, p, sc};
  const int m1[3] = {3, 4, 9}, m2[3] = {3, 4, 6};
  for (int q = 0; q < 3; ++q) {
    if (q == 2 && !c->prm.scalar) break;
    PTC_TRY(forward(c, rest[q], S.d_fa));
    P = SpecIn{};
    P.a = S.d_fa;
    if (S.on1d) PTC_TRY(spec_1d(c, P, kEnergy, m1[q]));
    if (S.on2d) PTC_TRY(spec_2d(c, S.d_fa, S.d_fa, m2[q], 1, 1.0));
  }
  ++S.nspectime;
  return PTC_OK;
}

// The accumulators to pageable host memory: pieces of kSpecStage bytes by way of
// two pinned halves, the next piece on its way while this one is copied out (14 MB
// at 512x128x256 with two rows of 2-D spectra: 1030 us a read through the
// runtime's own staging, now 830, of which 520 are the copy into fresh pages).
struct HostPiece {
  char *dst;
  const char *src;
  size_t n;
};
static int read_back(ptc_ctx *c, const std::vector<HostPiece> &pieces) {
  SpectraState &S = c->spec;
  auto fetch = [&](size_t q) -> int {
    PTC_HIP(hipMemcpyAsync(S.h_stage[q & 1], pieces[q].src, pieces[q].n, hipMemcpyDeviceToHost, c->stream));
    PTC_HIP(hipEventRecord(S.stage_ev[q & 1], c->stream));
    return PTC_OK;
  };
  if (!pieces.empty()) PTC_TRY(fetch(0));
  for (size_t q = 0; q < pieces.size(); ++q) {
    if (q + 1 < pieces.size()) PTC_TRY(fetch(q + 1));
    PTC_HIP(hipEventSynchronize(S.stage_ev[q & 1]));
    std::memcpy(pieces[q].dst, S.h_stage[q & 1], pieces[q].n);
  }
  return PTC_OK;
}

// The accumulated sums (not yet divided by nSpectime); reset zeroes them as
// the reference does after writing (src/m_FlowCase.f90:943-947).
int spectra_read(ptc_ctx *c, double *sx, double *sz, double *s2, int *nspectime, int reset) {
  SpectraState &S = c->spec;
  PTC_CHECK(S.ready, PTC_E_STATE, "spectra: call ptc_init_spectra first");
  std::vector<HostPiece> pieces;
  auto want = [&](double *dst, const double *src, size_t n) {
    for (size_t o = 0; o < n * sizeof(double); o += kSpecStage)
      pieces.push_back(HostPiece{reinterpret_cast<char *>(dst) + o, reinterpret_cast<const char *>(src) + o,
                                 std::min(kSpecStage, n * sizeof(double) - o)});
  };
  if (sx && S.on1d) want(sx, S.d_x, n1d_x(c));
  if (sz && S.on1d) want(sz, S.d_z, n1d_z(c));
  if (s2 && S.on2d) want(s2, S.d_2d, n2d(c));
  PTC_TRY(read_back(c, pieces));
  PTC_HIP(hipStreamSynchronize(c->stream));
  if (nspectime) *nspectime = S.nspectime;
  if (reset) {
    if (S.on1d) {
      PTC_TRY(fill_device(c, S.d_x, (long long)n1d_x(c), 0.0));
      PTC_TRY(fill_device(c, S.d_z, (long long)n1d_z(c), 0.0));
    }
    if (S.on2d) PTC_TRY(fill_device(c, S.d_2d, (long long)n2d(c), 0.0));
    S.nspectime = 0;
  }
  return PTC_OK;
}

}  // namespace ptc
