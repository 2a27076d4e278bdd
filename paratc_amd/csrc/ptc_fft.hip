// ptc_fft.hip -- FFT passes of the Poisson solve for any transform length.
//
// Replaces the FFTW r2r plans of the reference (R2HC / HC2R along x with
// stride 1 and along z with stride nx*ny, src/m_Poisson.f90:180-244) by two
// kernels that each make one read and one write pass over HBM:
//
//  * x pass: a real line of nx doubles is read as nx/2 complex pairs
//    z_m = x_{2m} + i x_{2m+1}, transformed with a complex FFT of length
//    h = nx/2 and unpacked to X_k, k = 0..h (the half spectrum).  The inverse
//    packs X_k back and applies the inverse FFT; HC2R(R2HC(x)) = nx x as in
//    FFTW, and the final 1/(nx nz) of the reference (normfft,
//    src/m_Poisson.f90:48,448) is applied on the store.
//  * z pass: complex FFTs of length nz on tiles of T consecutive kx columns,
//    so every global access moves T*16 contiguous bytes per z plane.
//
// The lengths that ptc_fft2.hip compiles for go there; these kernels take the
// radix plan at run time.  Every stage of a line has one butterfly per thread:
// its R inputs are loaded, transformed by a DFT whose radix is a compile-time
// constant (a switch on the plan's radix, uniform over the launch) and stored,
// in registers (two forms of workgroups of up to 1024 threads, held to 128
// VGPRs, spill: radix 15, 24-25 of them, for lines of 3375 and 3675 values only,
// and the x pass that forms the source in lines of more than 256 threads, 160:
// see poisson_div_fusable); the first stage reads HBM
// and the last one writes it, LDS carries the exchanges between them.  A line
// takes G = n / (smallest radix) threads; radices of 2 to 10 with as few and
// as even factors as the length allows (fft_make_len) keep the threads busy in
// every stage: 150 = 6 * 5 * 5, 180 = 6 * 6 * 5, 90 = 10 * 9.  The division
// by the span of a stage is a multiplication with a 32-bit reciprocal.  At
// 360 x 90 x 150 (80 MB moved per pass, all of it in the last-level cache, whence a
// copy of that size moves 6.8 TB/s) the four passes take 23-25 us each, 3.3 TB/s,
// at three to four waves per SIMD, where kernels that staged several run-time
// butterflies per thread in private memory took 52-55 us (solve 221 -> 102 us).
#include <cmath>
#include <cstring>

#include "ptc_dft.hpp"

namespace ptc {

using f2::cadd;
using f2::cmul;
using f2::csub;

// ---- one stage of a line: butterfly b = g of the n / R it has --------------
// x[b + r n/R] -> times w^(r k step), k = b mod span -> DFT -> x[(b div span)
// span R + k + r span].  SYNC: a barrier between the loads and the stores
// (both go to the same LDS line).  The powers of the twiddle step by w^4 from
// the first four, at most three products deep.
template <int R, bool INV, bool SYNC, class Load, class Store>
__device__ __forceinline__ void rt_butterfly(const FftLen &L, int s, int g, bool act, const Load &load,
                                             const Store &store) {
  const int nb = L.n / R, span = L.span[s];
  const bool on = act && g < nb;
  const int q = span > 1 ? (int)__umulhi((unsigned)g, L.magic[s]) : g;
  const int k = g - q * span;
  double2 w1 = make_double2(1.0, 0.0), v[R];
  if (on) {
    if (span > 1) {
      w1 = L.tw[k * L.step[s]];
      if (INV) w1.y = -w1.y;
    }
#pragma unroll
    for (int r = 0; r < R; ++r) v[r] = load(g + r * nb);
  }
  if (SYNC) __syncthreads();
  if (on) {
    if (span > 1) {
      double2 w[4];
      w[0] = w1;
      w[1] = cmul(w1, w1);
      w[2] = cmul(w[1], w1);
      w[3] = cmul(w[1], w[1]);
      const double2 w4 = w[3];
#pragma unroll
      for (int r = 1; r < R; ++r) {
        v[r] = cmul(v[r], w[(r - 1) % 4]);
        if (r + 4 < R) w[(r - 1) % 4] = cmul(w[(r - 1) % 4], w4);
      }
    }
    f2::Dft<R, INV>::run(v);
    const int d = q * span * R + k;
#pragma unroll
    for (int r = 0; r < R; ++r) store(d + r * span, v[r]);
  }
}

// RMAX: largest radix of the plans this instantiation runs (its code holds the
// registers of that radix whatever the plan)
template <int RMAX, bool INV, bool SYNC, class Load, class Store>
__device__ __forceinline__ void rt_stage(const FftLen &L, int s, int g, bool act, const Load &load,
                                         const Store &store) {
#define PTC_RADIX(R) \
  case R: rt_butterfly<R, INV, SYNC>(L, s, g, act, load, store); break;
  switch (L.radix[s]) {
    PTC_RADIX(2)
    PTC_RADIX(3)
    PTC_RADIX(4)
    PTC_RADIX(5)
    PTC_RADIX(6)
    PTC_RADIX(7)
    PTC_RADIX(8)
    PTC_RADIX(9)
    PTC_RADIX(10)
    default:
      if constexpr (RMAX > 10) {
        if (L.radix[s] == 15) rt_butterfly<15, INV, SYNC>(L, s, g, act, load, store);
      }
      break;
  }
#undef PTC_RADIX
}

// LDS slot of element m of an x line: one padding slot per 2^pad elements
__device__ __forceinline__ int rt_pad(int m, int pad) { return m + (m >> pad); }

// ---- x pass, forward: rows j = 1..ny of src -> half spectra in spec ----------
// nl lines per workgroup, G threads each; line q = (j - 1) + ny k, spec[q pitch +
// kx], kx = 0..h, zero to pitch.  DIV: the rows are formed from the velocities
// (div_pair) instead of read, their lines in tiles of tj x tk (line_tile; runs
// of two tiles' workgroups on one XCD) as the specialised pass orders them;
// each workgroup writes its maximum |divergence| to dv.part[blockIdx.x].
template <bool DIV, bool STREAM, int MAXT, int RMAX>
__global__ void __launch_bounds__(MAXT) k_fft_x_fwd(const double *__restrict__ src, double2 *__restrict__ spec,
                                                     FftLen L, const double2 *__restrict__ wx, int ny, int nz,
                                                     int nl, int pad, int pitch, long long rowlen, DivSrc dv, Geo geo,
                                                     int tj, int tk) {
  extern __shared__ double2 lds[];
  const int h = L.n, G = L.threads;
  const int l = threadIdx.x / G, g = threadIdx.x - l * G;
  const int tt = tj * tk;
  const int wb = DIV ? xcd_run((int)blockIdx.x, (int)gridDim.x, tt >= nl ? 2 * tt / nl : 1) : (int)blockIdx.x;
  const unsigned q = (unsigned)wb * nl + l;
  const bool live = l < nl && q < (unsigned)ny * nz;
  const LineAt at0 = line_at<DIV>(live ? q : 0, ny, nz, tj, tk);
  const long long jl = at0.j, k = at0.k;
  double2 *ls = lds + (l < nl ? l : 0) * (rt_pad(h - 1, pad) + 2);
  const double2 *row = reinterpret_cast<const double2 *>(src + rowlen * (jl + 1 + (long long)(ny + 2) * k));
  double dmax = 0.0;
  auto load0 = [&](int m) {
    if constexpr (DIV) return div_pair(dv, geo, h, ny, nz, rowlen, jl, k, m, dmax);
    else return f2::ld2x<STREAM>(row[m]);
  };
  auto at = [&](int m) { return ls[rt_pad(m, pad)]; };
  auto put = [&](int m, double2 v) { ls[rt_pad(m, pad)] = v; };
  rt_stage<RMAX, false, false>(L, 0, g, live, load0, put);
  __syncthreads();
  for (int s = 1; s < L.nstage; ++s) {
    rt_stage<RMAX, false, true>(L, s, g, live, at, put);
    __syncthreads();
  }
  if (live) {
    // X_k = (S_k - i w^k D_k) / 2, S_k, D_k = Z_k +- conj Z_{h-k}; four values'
    // twiddles are loaded before the first is used
    double2 *out = spec + (jl + (long long)ny * k) * pitch;
    for (int k0 = g; k0 < pitch; k0 += 4 * G) {
      double2 w[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) w[u] = wx[min(k0 + u * G, h)];
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const int kx = k0 + u * G;
        if (kx >= pitch) break;
        double2 X = make_double2(0.0, 0.0);
        if (kx <= h) {
          const double2 zk = at(kx == h ? 0 : kx);
          double2 zc = at(kx == 0 ? 0 : h - kx);
          zc.y = -zc.y;
          const double2 sm = cadd(zk, zc), wd = cmul(w[u], csub(zk, zc));
          X = make_double2(0.5 * (sm.x + wd.y), 0.5 * (sm.y - wd.x));
        }
        f2::st2x<STREAM>(out[kx], X);
      }
    }
  }
  if constexpr (DIV) {
    const double dm = block_max_tree(dmax, reinterpret_cast<double *>(lds));
    if (threadIdx.x == 0) dv.part[blockIdx.x] = dm;
  }
}

// ---- x pass, inverse: half spectra -> real rows, scaled -----------------------
// ghost: the rows j = 1 and j = ny also go to the Neumann ghost rows
// (SetBC_and_UpdateHalo_pr, src/m_BC_and_Halo.f90:115-120)
template <bool STREAM, int MAXT, int RMAX>
__global__ void __launch_bounds__(MAXT) k_fft_x_inv(const double2 *__restrict__ spec, double *__restrict__ dst,
                                                     FftLen L, const double2 *__restrict__ wx, int ny, int nz,
                                                     int nl, int pad, int pitch, long long rowlen, double scale,
                                                     int ghost) {
  extern __shared__ double2 lds[];
  const int h = L.n, G = L.threads;
  const int l = threadIdx.x / G, g = threadIdx.x - l * G;
  const unsigned q = blockIdx.x * nl + l;
  const bool live = l < nl && q < (unsigned)ny * nz;
  const LineAt at0 = line_at<false>(live ? q : 0, ny, nz, 1, 1);
  const long long jl = at0.j, k = at0.k;
  double2 *ls = lds + (l < nl ? l : 0) * (rt_pad(h, pad) + 1);
  auto at = [&](int m) { return ls[rt_pad(m, pad)]; };
  auto put = [&](int m, double2 v) { ls[rt_pad(m, pad)] = v; };
  if (live) {
    // the line's h+1 values go through LDS once; eight loads in flight
    // (indices past h repeat element h)
    const double2 *in = spec + (jl + (long long)ny * k) * pitch;
    for (int m0 = g; m0 <= h; m0 += 8 * G) {
      double2 v[8];
#pragma unroll
      for (int u = 0; u < 8; ++u) v[u] = f2::ld2x<STREAM>(in[min(m0 + u * G, h)]);
#pragma unroll
      for (int u = 0; u < 8; ++u) put(min(m0 + u * G, h), v[u]);
    }
  }
  __syncthreads();
  // X_m + conj X_{h-m} + i conj(w^m) (X_m - conj X_{h-m})
  auto load0 = [&](int m) {
    const double2 xk = at(m);
    double2 xc = at(h - m), w = wx[m];
    xc.y = -xc.y;
    w.y = -w.y;
    const double2 sm = cadd(xk, xc), wd = cmul(w, csub(xk, xc));
    return make_double2(sm.x - wd.y, sm.y + wd.x);
  };
  double2 *row = reinterpret_cast<double2 *>(dst + rowlen * (jl + 1 + (long long)(ny + 2) * k));
  auto store_out = [&](int m, double2 v) {
    const double2 x = make_double2(v.x * scale, v.y * scale);
    f2::st2x<STREAM>(row[m], x);
    if (ghost && jl == 0) f2::st2x<STREAM>(row[m - h], x);
    if (ghost && jl == ny - 1) f2::st2x<STREAM>(row[m + h], x);
  };
  if (L.nstage == 1) {
    rt_stage<RMAX, true, true>(L, 0, g, live, load0, store_out);
    return;
  }
  rt_stage<RMAX, true, true>(L, 0, g, live, load0, put);
  __syncthreads();
  for (int s = 1; s + 1 < L.nstage; ++s) {
    rt_stage<RMAX, true, true>(L, s, g, live, at, put);
    __syncthreads();
  }
  rt_stage<RMAX, true, false>(L, L.nstage - 1, g, live, at, store_out);
}

// ---- z pass: complex FFT of length nz on T columns of one plane ---------------
// thread = g T + column; column tile and plane from the XCD-grouped workgroup
// index, so that the tiles sharing a 128-byte row segment use one L2
template <bool INV, int MAXT>
__global__ void __launch_bounds__(MAXT) k_fft_z(double2 *__restrict__ spec, FftLen L, int ny, int pitch, int T,
                                                 int ntile) {
  extern __shared__ double2 lds[];
  const int col = threadIdx.x & (T - 1), g = threadIdx.x / T;
  const bool act = g < L.threads;
  const long long zs = (long long)pitch * ny;
  const int w = xcd_run((int)blockIdx.x, (int)gridDim.x, T < 8 ? 8 / T : 1);
  const int tile = w % ntile, jj = w / ntile;
  double2 *base = spec + (long long)jj * pitch + (long long)tile * T + col;
  auto load0 = [&](int m) { return base[m * zs]; };
  auto store_out = [&](int m, double2 v) { base[m * zs] = v; };
  auto at = [&](int m) { return lds[m * T + col]; };
  auto put = [&](int m, double2 v) { lds[m * T + col] = v; };
  if (L.nstage == 1) {
    rt_stage<10, INV, false>(L, 0, g, act, load0, store_out);
    return;
  }
  rt_stage<10, INV, false>(L, 0, g, act, load0, put);
  __syncthreads();
  for (int s = 1; s + 1 < L.nstage; ++s) {
    rt_stage<10, INV, true>(L, s, g, act, at, put);
    __syncthreads();
  }
  rt_stage<10, INV, false>(L, L.nstage - 1, g, act, at, store_out);
}

// ---- host side -----------------------------------------------------------

// The factorisation of n into radices 2..10 with the fewest factors, of those
// the one whose smallest factor is largest (the fewest threads per line, so the
// fewest idle in the other stages).  Radices of 12 to 16 would take a stage out
// of many lengths, but 194 VGPRs instead of 128, and lost.  most = 15: also
// radix 15, for the odd lengths (3375, 3675) whose lines would otherwise take
// more than 1024 threads.
static void best_radices(int m, int most, int *cur, int nc, int *best, int *nbest) {
  if (m == 1) {
    const bool fewer = nc < *nbest;
    // cur descends, so its last factor is the smallest
    if (fewer || (nc == *nbest && cur[nc - 1] > best[nc - 1])) {
      std::memcpy(best, cur, sizeof(int) * nc);
      *nbest = nc;
    }
    return;
  }
  if (nc + 1 > *nbest || nc >= kFftMaxStages) return;
  for (int r : {15, 10, 9, 8, 7, 6, 5, 4, 3, 2})
    if (r <= most && m % r == 0) {
      cur[nc] = r;
      best_radices(m / r, r, cur, nc + 1, best, nbest);
    }
}

int fft_make_len(int n, FftLen *L) {
  std::memset(L, 0, sizeof(*L));
  L->n = n;
  int m = n;
  for (int f : {2, 3, 5, 7})
    while (m % f == 0) m /= f;
  if (m != 1 || n < 2) {
    set_error("FFT length " + std::to_string(n) + " has a prime factor other than 2, 3, 5, 7");
    return PTC_E_UNSUPPORTED;
  }
  int cur[kFftMaxStages], best[kFftMaxStages], nbest = kFftMaxStages + 1;
  best_radices(n, 10, cur, 0, best, &nbest);
  if (nbest <= kFftMaxStages && n / best[nbest - 1] > 1024) {
    nbest = kFftMaxStages + 1;
    best_radices(n, 15, cur, 0, best, &nbest);
  }
  if (nbest > kFftMaxStages) {
    set_error("FFT length " + std::to_string(n) + " has too many factors");
    return PTC_E_UNSUPPORTED;
  }
  L->nstage = nbest;
  int span = 1;
  for (int s = 0; s < nbest; ++s) {
    L->radix[s] = best[s];
    L->span[s] = span;
    // floor(b / span) = umulhi(b, ceil(2^32 / span)) for b < 2^16, 1 < span < 2^16
    L->magic[s] = span > 1 ? (unsigned)(((1ull << 32) + span - 1) / span) : 0u;
    span *= best[s];
    L->step[s] = n / span;
  }
  L->threads = n / best[nbest - 1];
  return PTC_OK;
}

// launch shape of the x passes: lines per workgroup (about 256 threads), LDS
// padding and bytes; false if a line's threads or the launch's bytes do not fit.
// Lines that pass pad_cap bytes with the padding go without it: a line holds n + 1
// slots then (the inverse keeps X_0 .. X_n), at n = 4096 16 bytes over 64 KB.
bool fft_x_shape(const FftLen &L, size_t pad_cap, size_t lds_limit, int *lines, int *threads, int *pad, size_t *lds) {
  if (L.threads > 1024) return false;
  *lines = std::max(1, 256 / L.threads);
  *threads = (*lines * L.threads + 63) / 64 * 64;
  *pad = 3;
  size_t slots = (size_t)L.n + L.n / 8 + 1;
  if (sizeof(double2) * slots > pad_cap) {
    *pad = 30;
    slots = (size_t)L.n + 1;
  }
  // room for the divergence maximum's tree, one double per thread
  *lds = std::max(sizeof(double2) * slots * *lines, sizeof(double) * (size_t)*threads);
  return *lds <= lds_limit;
}

// columns per z workgroup: the largest power of two up to `most` whose tile
// fits LDS and whose workgroup fits 1024 threads
int fft_z_tile(const FftLen &L, size_t lds_cap, int most) {
  int T = most;
  while (T > 1 && (sizeof(double2) * (size_t)L.n * T > lds_cap || (long long)T * L.threads > 1024)) T /= 2;
  return T;
}

long long fft_x_div_blocks(const ptc_ctx *c, int nj) {
  const PoissonPlan &P = c->pp;
  if (P.x_fast || !P.ready) return fft2_x_div_blocks(c, nj);
  return ((long long)nj * c->nz + P.x_lines - 1) / P.x_lines;
}

template <bool DIV, bool STREAM, int MAXT, int RMAX>
static void x_fwd_rt(ptc_ctx *c, const double *src, double2 *spec, const DivSrc &dv) {
  PoissonPlan &P = c->pp;
  int tj = 1, tk = 1;
  if (DIV) line_tile(c->ny, c->nz, &tj, &tk);
  const long long nlines = (long long)c->ny * c->nz;
  hipLaunchKernelGGL((k_fft_x_fwd<DIV, STREAM, MAXT, RMAX>), dim3((unsigned)((nlines + P.x_lines - 1) / P.x_lines)),
                     dim3(P.x_threads), P.x_lds, c->stream, src, spec, P.fx, P.d_wx, c->ny, c->nz, P.x_lines, P.x_pad, P.pitch,
                     (long long)c->nx, dv, c->geo, tj, tk);
}

template <bool DIV, bool STREAM>
static void x_fwd_launch_s(ptc_ctx *c, const double *src, double2 *spec, const DivSrc &dv) {
  if (!DIV && c->pp.fx.radix[0] > 10) x_fwd_rt<false, STREAM, 1024, 15>(c, src, spec, dv);
  else if (c->pp.x_threads > 256) x_fwd_rt<DIV, STREAM, 1024, 10>(c, src, spec, dv);
  else x_fwd_rt<DIV, STREAM, 256, 10>(c, src, spec, dv);
}

template <bool DIV>
static int x_fwd_launch(ptc_ctx *c, const double *src, double2 *spec, const DivSrc &dv) {
  if (c->pp.stream) x_fwd_launch_s<DIV, true>(c, src, spec, dv);
  else x_fwd_launch_s<DIV, false>(c, src, spec, dv);
  PTC_HIP(hipGetLastError());
  return PTC_OK;
}

int launch_fft_x_fwd(ptc_ctx *c, const double *src, void *spec, bool f64) {
  if (c->pp.x_fast) return fft2_x_fwd(c, src, spec, 0, c->ny, f64);
  return x_fwd_launch<false>(c, src, static_cast<double2 *>(spec), DivSrc{});
}

int launch_fft_x_fwd_div(ptc_ctx *c, const DivSrc &div, void *spec) {
  if (c->pp.x_fast) return fft2_x_fwd(c, nullptr, spec, 0, c->ny, false, &div);
  return x_fwd_launch<true>(c, nullptr, static_cast<double2 *>(spec), div);
}

template <bool STREAM, int MAXT, int RMAX>
static void x_inv_rt(ptc_ctx *c, const double2 *spec, double *dst, double scale, bool ghost) {
  PoissonPlan &P = c->pp;
  const long long nlines = (long long)c->ny * c->nz;
  hipLaunchKernelGGL((k_fft_x_inv<STREAM, MAXT, RMAX>), dim3((unsigned)((nlines + P.x_lines - 1) / P.x_lines)),
                     dim3(P.x_threads), P.x_lds, c->stream, spec, dst, P.fx, P.d_wx, c->ny, c->nz, P.x_lines, P.x_pad,
                     P.pitch, (long long)c->nx, scale, ghost ? 1 : 0);
}

template <bool STREAM>
static void x_inv_launch(ptc_ctx *c, const double2 *spec, double *dst, double scale, bool ghost) {
  if (c->pp.fx.radix[0] > 10) x_inv_rt<STREAM, 1024, 15>(c, spec, dst, scale, ghost);
  else if (c->pp.x_threads > 256) x_inv_rt<STREAM, 1024, 10>(c, spec, dst, scale, ghost);
  else x_inv_rt<STREAM, 256, 10>(c, spec, dst, scale, ghost);
}

// ghost: also fill the Neumann ghost rows
int launch_fft_x_inv(ptc_ctx *c, const void *spec_, double *dst, double scale, bool acc, bool ghost) {
  if (c->pp.x_fast) return fft2_x_inv(c, spec_, dst, scale, 0, c->ny, acc, ghost);
  PTC_CHECK(!acc, PTC_E_UNSUPPORTED, "accumulating x-inverse needs the specialised kernels");
  const double2 *spec = static_cast<const double2 *>(spec_);
  if (c->pp.stream) x_inv_launch<true>(c, spec, dst, scale, ghost);
  else x_inv_launch<false>(c, spec, dst, scale, ghost);
  PTC_HIP(hipGetLastError());
  return PTC_OK;
}

int launch_fft_z(ptc_ctx *c, void *spec_, bool inverse, bool f64) {
  if (c->pp.z_fast) return fft2_z(c, spec_, inverse, 0, c->ny, f64);
  PoissonPlan &P = c->pp;
  double2 *spec = static_cast<double2 *>(spec_);
  const size_t lds = sizeof(double2) * (size_t)P.fz.n * P.ztile;
  const int ntile = P.pitch / P.ztile, nt = P.fz.threads * P.ztile;
  const dim3 grid((unsigned)(ntile * c->ny)), blk((unsigned)((nt + 63) / 64 * 64));
#define PTC_Z(INV, MAXT) \
  hipLaunchKernelGGL((k_fft_z<INV, MAXT>), grid, blk, lds, c->stream, spec, P.fz, c->ny, P.pitch, P.ztile, ntile)
  if (inverse && nt > 256) PTC_Z(true, 1024);
  else if (inverse) PTC_Z(true, 256);
  else if (nt > 256) PTC_Z(false, 1024);
  else PTC_Z(false, 256);
#undef PTC_Z
  PTC_HIP(hipGetLastError());
  return PTC_OK;
}

}  // namespace ptc
