// ptc_fft2.hip -- compile-time specialised, register-resident FFT passes.
//
// For the transform lengths of the production grids the radix plan, the
// number of stages and the threads per line are compile-time constants, so
// every butterfly lives in registers and no private (scratch) memory is used.
// Stage 0 reads its inputs straight from HBM and the last stage writes its
// outputs straight to HBM; LDS only carries the exchanges between stages.
// The algorithm is the same self-sorting Stockham transform as the run-time
// length kernels of ptc_fft.hip (the path for other lengths):
//
//   stage with radix R after a span Ns:  butterfly b reads x[b + r N/R],
//   multiplies by w^(r (b mod Ns) N/(Ns R)), applies the R-point DFT and
//   writes x[(b div Ns) Ns R + (b mod Ns) + r Ns].
//
// Twiddles: w^e for the first power comes from the host FP64 table; the
// higher powers of the same stage are formed by complex products (at most six
// products, error ~ 7 ulp), which replaces R-1 table loads per butterfly.
#include <algorithm>

#include "ptc_dft.hpp"

namespace ptc {

namespace f2 {

// ---- compile-time radix plan: 8s first, then 4 or 2, then 9, 3, 5, 7 ----
struct PlanC {
  int ns;
  int r[12];
};

constexpr PlanC make_plan(int n) {
  PlanC p{0, {0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0}};
  int m = n;
  while (m % 8 == 0) { p.r[p.ns++] = 8; m /= 8; }
  if (m % 4 == 0) { p.r[p.ns++] = 4; m /= 4; }
  if (m % 2 == 0) { p.r[p.ns++] = 2; m /= 2; }
  while (m % 9 == 0) { p.r[p.ns++] = 9; m /= 9; }
  while (m % 3 == 0) { p.r[p.ns++] = 3; m /= 3; }
  while (m % 5 == 0) { p.r[p.ns++] = 5; m /= 5; }
  while (m % 7 == 0) { p.r[p.ns++] = 7; m /= 7; }
  if (m != 1) p.ns = -1;
  return p;
}

constexpr int plan_rmax(int n) {
  PlanC p = make_plan(n);
  int mx = 1;
  for (int s = 0; s < p.ns; ++s) mx = p.r[s] > mx ? p.r[s] : mx;
  return mx;
}

constexpr int plan_span(int n, int s) {  // product of the radices before stage s
  PlanC p = make_plan(n);
  int v = 1;
  for (int q = 0; q < s; ++q) v *= p.r[q];
  return v;
}

// LDS padding of one line: one slot per 8 elements
__device__ __forceinline__ int pad8(int m) { return m + (m >> 3); }
constexpr int padded(int n) { return n + n / 8 + 1; }

// ---- one stage for the G threads of a line; Load(m) / Store(m, v) address the
//      line's elements.  SYNC: a barrier separates this stage's loads from its
//      stores (needed when both go to the same LDS buffer). ----
// butterflies per thread of stage S (at most 4: G = N / rmax, radix >= 2)
template <int N, int S, int G>
constexpr int stage_bpt() {
  return (N / make_plan(N).r[S] + G - 1) / G;
}

// The first twiddle w1 of each butterfly a thread runs in stage S, read from
// the table ahead of the transform (it does not depend on the data), so no
// stage waits on a global load.
template <int N, int S, int G, bool INV>
__device__ __forceinline__ void stage_twiddles(int g, const double2 *__restrict__ tw, double2 (&w)[4]) {
  constexpr PlanC P = make_plan(N);
  constexpr int R = P.r[S];
  constexpr int NS = plan_span(N, S);
  constexpr int NB = N / R;
  constexpr int BPT = stage_bpt<N, S, G>();
  static_assert(BPT <= 4, "at most four butterflies per thread");
#pragma unroll
  for (int i = 0; i < BPT; ++i) {
    const int b = g + i * G;
    const int k = (BPT * G == NB || b < NB) ? b % NS : 0;
    w[i] = NS > 1 ? tw[k * (N / (NS * R))] : make_double2(1.0, 0.0);
    if (INV) w[i].y = -w[i].y;
  }
}

// stage S's inputs of one thread: v[i][r] = element b + r * NB of butterfly
// b = g + i * G
template <int N, int S, int G>
using StageRegs = double2[stage_bpt<N, S, G>()][make_plan(N).r[S]];

template <int N, int S, int G, class Load>
__device__ __forceinline__ void stage_load(int g, const Load &load, StageRegs<N, S, G> &v) {
  constexpr int R = make_plan(N).r[S];
  constexpr int NB = N / R;
  constexpr int BPT = stage_bpt<N, S, G>();
#pragma unroll
  for (int i = 0; i < BPT; ++i) {
    const int b = g + i * G;
    if (BPT * G == NB || b < NB) {
#pragma unroll
      for (int r = 0; r < R; ++r) v[i][r] = load(b + r * NB);
    }
  }
}

template <int N, int S, int G, bool INV, class Store>
__device__ __forceinline__ void stage_exec(int g, const double2 (&wpre)[4], StageRegs<N, S, G> &v,
                                           const Store &store) {
  constexpr int R = make_plan(N).r[S];
  constexpr int NS = plan_span(N, S);
  constexpr int NB = N / R;
  constexpr int BPT = stage_bpt<N, S, G>();
#pragma unroll
  for (int i = 0; i < BPT; ++i) {
    const int b = g + i * G;
    if (BPT * G == NB || b < NB) {
      const int k = b % NS;
      if (NS > 1) {
        const double2 w1 = wpre[i];
        double2 w = w1;
#pragma unroll
        for (int r = 1; r < R; ++r) {
          v[i][r] = cmul(v[i][r], w);
          if (r + 1 < R) w = cmul(w, w1);
        }
      }
      Dft<R, INV>::run(v[i]);
      const int idxD = (b / NS) * NS * R + k;
#pragma unroll
      for (int r = 0; r < R; ++r) store(idxD + r * NS, v[i][r]);
    }
  }
}

template <int N, int S, int G, bool INV, bool SYNC, class Load, class Store>
__device__ __forceinline__ void stage(int g, const double2 (&wpre)[4], const Load &load, const Store &store) {
  StageRegs<N, S, G> v;
  stage_load<N, S, G>(g, load, v);
  if (SYNC) __syncthreads();
  stage_exec<N, S, G, INV>(g, wpre, v, store);
}

// Full transform of one line group.  Stage 0 loads through load0, the last
// stage stores through storeL; intermediate data lives in LDS through lds(m).
// LOAD0_LDS: load0 itself reads the LDS buffer, so stage 0 needs a barrier
// between its loads and its stores.
// the first twiddles of every stage a thread runs
template <int N, int G, bool INV>
__device__ __forceinline__ void load_twiddles(int g, const double2 *__restrict__ tw, double2 (&W)[7][4]) {
  constexpr PlanC P = make_plan(N);
  static_assert(P.ns <= 7, "too many stages");
  stage_twiddles<N, 0, G, INV>(g, tw, W[0]);
  if constexpr (P.ns > 1) stage_twiddles<N, (P.ns > 1 ? 1 : 0), G, INV>(g, tw, W[1]);
  if constexpr (P.ns > 2) stage_twiddles<N, (P.ns > 2 ? 2 : 0), G, INV>(g, tw, W[2]);
  if constexpr (P.ns > 3) stage_twiddles<N, (P.ns > 3 ? 3 : 0), G, INV>(g, tw, W[3]);
  if constexpr (P.ns > 4) stage_twiddles<N, (P.ns > 4 ? 4 : 0), G, INV>(g, tw, W[4]);
  if constexpr (P.ns > 5) stage_twiddles<N, (P.ns > 5 ? 5 : 0), G, INV>(g, tw, W[5]);
  if constexpr (P.ns > 6) stage_twiddles<N, (P.ns > 6 ? 6 : 0), G, INV>(g, tw, W[6]);
}

// Stages 1 .. ns-1 of a transform whose stage 0 has stored into LDS (and a
// barrier has passed); the last stage stores through storeL.
template <int N, int G, bool INV, class LdsAt, class StoreL>
__device__ __forceinline__ void run_rest(int g, const double2 (&W)[7][4], const LdsAt &lds, const StoreL &storeL) {
  constexpr PlanC P = make_plan(N);
  static_assert(P.ns >= 2, "a single-stage transform has no later stages");
  auto ldsload = [&](int m) { return lds(m); };
  auto ldsstore = [&](int m, double2 v) { lds(m) = v; };
  if constexpr (P.ns > 2) {
    stage<N, 1, G, INV, true>(g, W[1], ldsload, ldsstore);
    __syncthreads();
  }
  if constexpr (P.ns > 3) {
    stage<N, 2, G, INV, true>(g, W[2], ldsload, ldsstore);
    __syncthreads();
  }
  if constexpr (P.ns > 4) {
    stage<N, 3, G, INV, true>(g, W[3], ldsload, ldsstore);
    __syncthreads();
  }
  if constexpr (P.ns > 5) {
    stage<N, 4, G, INV, true>(g, W[4], ldsload, ldsstore);
    __syncthreads();
  }
  if constexpr (P.ns > 6) {
    stage<N, 5, G, INV, true>(g, W[5], ldsload, ldsstore);
    __syncthreads();
  }
  stage<N, P.ns - 1, G, INV, true>(g, W[P.ns - 1], ldsload, storeL);
}

// the whole transform with the first twiddles already in registers
template <int N, int G, bool INV, bool LOAD0_LDS = false, class Load0, class LdsAt, class StoreL>
__device__ __forceinline__ void run_fft_w(int g, const double2 (&W)[7][4], const Load0 &load0, const LdsAt &lds,
                                          const StoreL &storeL) {
  constexpr PlanC P = make_plan(N);
  if constexpr (P.ns == 1) {
    stage<N, 0, G, INV, false>(g, W[0], load0, storeL);
  } else {
    auto ldsstore = [&](int m, double2 v) { lds(m) = v; };
    stage<N, 0, G, INV, LOAD0_LDS>(g, W[0], load0, ldsstore);
    __syncthreads();
    run_rest<N, G, INV>(g, W, lds, storeL);
  }
}

template <int N, int G, bool INV, bool LOAD0_LDS = false, class Load0, class LdsAt, class StoreL>
__device__ __forceinline__ void run_fft(int g, const double2 *__restrict__ tw, const Load0 &load0, const LdsAt &lds,
                                        const StoreL &storeL) {
  double2 W[7][4];
  load_twiddles<N, G, INV>(g, tw, W);
  run_fft_w<N, G, INV, LOAD0_LDS>(g, W, load0, lds, storeL);
}

}  // namespace f2

// threads per line: the largest-radix stage has one butterfly per thread (a
// radix-9 stage counts as 8: its N/9 butterflies fit the N/8 threads of the
// radix-8 stages)
template <int N>
constexpr int f2_threads() {
  return N / (f2::plan_rmax(N) > 8 ? 8 : f2::plan_rmax(N));
}

// x-pass workgroup: about 64 threads for rows of up to 256 points, about 256 for
// longer ones (several lines each), or one line of G > 256 threads.  Short rows
// belong to small grids, whose few hundred workgroups of 256 threads leave CUs
// idle and fill the last round unevenly: RK substep 64x48x64 58.1 -> 55.1 us,
// 96x64x96 84.5 -> 83.0, 128x48x64 68.0 -> 66.4, 192x64x96 126.7 -> 123.8,
// 128x96x128 and 192x128x192 the same; rows of 512 points 1239 -> 1235 at 128.
template <int N>
constexpr int f2_xbase() {
  return N <= 128 ? 64 : 256;
}
// its threads at most
template <int N>
constexpr int f2_xblock() {
  return f2_threads<N>() > f2_xbase<N>() ? f2_threads<N>() : f2_xbase<N>();
}

// LDS layout of an x-pass line: one padding value after every 8 (bank
// spreading), after every 16 for the 4608-point lines, so that such a line
// (78 KB) leaves room for a second workgroup on the CU's 160 KB
template <int N>
__device__ __forceinline__ int xpad(int m) {
  return N == 4608 ? m + (m >> 4) : f2::pad8(m);
}
template <int N>
constexpr int xpadded() {
  return N == 4608 ? N + N / 16 + 1 : f2::padded(N);
}

// The half spectrum of a real row of 2N points from the N-point transform Z
// of its packed pairs (in ls): X_k = (S_k - i w^k D_k) / 2 with
// S_k = Z_k + conj Z_{N-k}, D_k = Z_k - conj Z_{N-k}, w = exp(-2 pi i / 2N);
// values past k = N (pitch padding) are zero.
template <int N, int G, bool STREAM, typename S>
__device__ __forceinline__ void x_untangle_store(int g, const double2 *ls, const double2 *__restrict__ wx,
                                                 S *__restrict__ out, int pitch) {
  // pitch <= N + 32: a thread stores at most NK values.  Their twiddles are
  // all loaded before the first is used, so the thread waits once on them
  // (a load per iteration waited on every load in flight, the next line's
  // prefetch included, once per value).
  constexpr int NK = (N + 32 + G - 1) / G;
  double2 w[NK];
#pragma unroll
  for (int t = 0; t < NK; ++t) w[t] = wx[min(g + t * G, N)];
#pragma unroll
  for (int t = 0; t < NK; ++t) {
    const int kx = g + t * G;
    if (kx >= pitch) break;
    double2 X = make_double2(0.0, 0.0);
    if (kx <= N) {
      const double2 zk = ls[xpad<N>(kx == N ? 0 : kx)];
      double2 zc = ls[xpad<N>(kx == 0 ? 0 : N - kx)];
      zc.y = -zc.y;
      const double2 s = f2::cadd(zk, zc), d = f2::csub(zk, zc);
      const double2 wd = f2::cmul(w[t], d);
      X = make_double2(0.5 * (s.x + wd.y), 0.5 * (s.y - wd.x));
    }
    f2::st2x<STREAM>(out[kx], X);
  }
}

// The inverse: element m of the N-point inverse transform's input from the
// half spectrum X (in ls): X_m + conj X_{N-m} + i conj(w^m) (X_m - conj X_{N-m}).
template <int N>
__device__ __forceinline__ double2 x_retangle(const double2 *ls, const double2 *__restrict__ wx, int m) {
  const double2 xk = ls[xpad<N>(m)];
  double2 xc = ls[xpad<N>(N - m)];
  xc.y = -xc.y;
  const double2 s = f2::cadd(xk, xc), d = f2::csub(xk, xc);
  double2 w = wx[m];
  w.y = -w.y;
  const double2 wd = f2::cmul(w, d);
  return make_double2(s.x - wd.y, s.y + wd.x);
}

// Waves per SIMD the one-shot x kernels are held to.  2304-point lines: 288
// threads and 41 KB of LDS, three workgroups (15 waves) per CU at four waves
// per SIMD (128 VGPRs; left alone the inverse takes 129 and two fit).
// 4608-point lines: 576 threads and 78 KB, two workgroups (18 waves) per CU
// at five (102 VGPRs).
template <int N>
constexpr int f2_x_min_waves() {
  return N == 2304 ? 4 : (N == 4608 ? 5 : 1);
}
// The residual-forming form holds twenty more loads per point pair: held to
// those bounds it spills 96-188 bytes per lane, so it takes the registers it
// needs (three waves per SIMD at most).
// The divergence by columns takes 130 VGPRs at 512-point rows and 117 at 1024 and
// is left alone: held to 128 the former spilled 7 and was slower (a step of
// 512x128x256 3736 us against 3721, 512x96x128 1429 against 1415).
template <int N, int SRC>
constexpr int f2_xfwd_min_waves() {
  return SRC >= 2 ? ((N == 2304 || N == 4608) ? 3 : 1) : f2_x_min_waves<N>();
}
// Planes a thread takes at a time where the divergence is formed by columns
// (1: pair by pair), and the lines of a workgroup then, whole groups of them.
template <int N>
constexpr int f2_div_planes() {
  constexpr int L = f2_threads<N>() <= f2_xbase<N>() ? f2_xbase<N>() / f2_threads<N>() : 1;
  return L >= 4 ? 4 : (L >= 2 ? 2 : 1);
}
template <int N>
constexpr int f2_div_lines() {
  constexpr int L = f2_threads<N>() <= f2_xbase<N>() ? f2_xbase<N>() / f2_threads<N>() : 1;
  return L / f2_div_planes<N>() * f2_div_planes<N>();
}
// Lines of one plane column in the column form of the residual (kXResCol), or
// 0 where the length has none: a workgroup's lines in groups of K consecutive
// planes of one row, N * lines a multiple of K times the threads (f2_xbase).
template <int N>
constexpr int f2_res_lines() {
  constexpr int L = f2_threads<N>() <= f2_xbase<N>() ? f2_xbase<N>() / f2_threads<N>() : 1;
  return L * f2_threads<N>() == f2_xbase<N>() ? (L % 8 == 0 ? 8 : (L == 4 ? 4 : 0)) : 0;
}

// ---- x forward: nlpb real rows of length 2N -> half spectra ---------------
// SRC = kXDiv: the rows are not read from src but formed from the velocities,
// as clcPrSrc does (div_value), by columns of planes where a workgroup holds two
// lines or more (f2_div_planes), else pair by pair.  Each workgroup then writes
// the maximum |divergence| over its rows to dv.part[blockIdx.x].
// SRC = kXRes: the rows are the refinement's FP64 residual f - L phi, in
// k_residual's operand order; each workgroup writes the sum of phi over its
// lines of row j = 1 to rs.psum[blockIdx.x].
// By columns and in workgroups of 64 threads (rows of up to 256 points) the RK
// substep of 64x48x64 took 55.1 us against 59.2, 192x64x96 123.8 against 127.4,
// 512x128x256 1234 against 1250; by columns alone 58.1, 126.6 and 1240.
// SRC = kXResCol: the same residual, formed by columns.  The direct form loads
// fifteen pairs per pair of points (five of its own row, six planes, two rows,
// f), 16 GB through L1 at 1024x256x512; here a thread forms one pair m of K
// consecutive planes, whose K + 6 planes it loads once, and reads the row
// neighbours from the lines' LDS: 5.5 (K = 4) or 4.75 (K = 8) loads a pair.
// 1022 -> 780 us there with FP32 spectra (2.1 GB in, 0.5 GB out; the shape of
// the tiles and f's caching hint move it by under 1 %: it waits on its two
// rounds of loads, at three waves per SIMD).
// Needs tk a multiple of K, so that no group of K lines leaves its row.
constexpr int kXPlain = 0, kXDiv = 1, kXRes = 2, kXResCol = 3;

// The residual of a workgroup's lines q0 .. q0+L-1 into their LDS rows (the
// column form).  Each thread takes the columns threadIdx.x + f2_xbase c: pair m of
// the K planes of one group of lines.  All the planes of its columns are in
// flight at once, then the rows above and below and f, one column after the
// other; edge rows load their own row for the missing one (the Neumann
// condition), so no load sits behind a branch.
template <int N, int K, bool STREAM>
__device__ __forceinline__ void res_columns(double2 *sh, const ResSrc &rs, const Geo &geo, int ny, int nz,
                                            long long rowlen, int j0, unsigned q0, unsigned nlines, int tj, int tk,
                                            double &psum) {
  constexpr double st0 = -1460.0 / 576.0, st1 = 783.0 / 576.0, st2 = -54.0 / 576.0, st3 = 1.0 / 576.0;
  constexpr int T = f2_xbase<N>(), L = T / f2_threads<N>();
  constexpr int NC = N * (L / K) / T;  // columns per thread
  static_assert(NC * T == N * (L / K), "whole columns");
  constexpr int PN = xpadded<N>();
  const long long pl = rowlen * (ny + 2);
  double2 z[NC][K + 6];
  long long base[NC];  // offset of the group's first line
  int mc[NC], gc[NC], jc[NC];
  bool ok[NC];
#pragma unroll
  for (int c = 0; c < NC; ++c) {
    const int col = (int)threadIdx.x + T * c;
    mc[c] = col % N;
    gc[c] = col / N;
    const unsigned q = q0 + gc[c] * K;
    ok[c] = q < nlines;
    const LineAt at = line_at<true>(ok[c] ? q : 0, 1, nz, tj, tk);
    const int jl = j0 + at.j, k = at.k;
    jc[c] = jl + 1;
    base[c] = rowlen * (jl + 1 + (long long)(ny + 2) * k);
#pragma unroll
    for (int s = 0; s < K + 6; ++s) {
      int kk = k - 3 + s;
      kk = kk < 0 ? kk + nz : (kk >= nz ? kk - nz : kk);
      z[c][s] = reinterpret_cast<const double2 *>(rs.phi + base[c] + (kk - k) * pl)[mc[c]];
    }
  }
#pragma unroll
  for (int c = 0; c < NC; ++c)
#pragma unroll
    for (int i = 0; i < K; ++i) sh[(gc[c] * K + i) * PN + xpad<N>(mc[c])] = z[c][3 + i];
  __syncthreads();
  double2 r[NC][K];
#pragma unroll
  for (int c = 0; c < NC; ++c) {
    const int m = mc[c], j = jc[c];
    const double am = geo.met[M_AM2PH * geo.nyh + j], ac = geo.met[M_AC2PH * geo.nyh + j],
                 ap = geo.met[M_AP2PH * geo.nyh + j];
    const int m1 = m - 1 < 0 ? m - 1 + N : m - 1, m2 = m - 2 < 0 ? m - 2 + N : m - 2;
    const int p1 = m + 1 >= N ? m + 1 - N : m + 1, p2 = m + 2 >= N ? m + 2 - N : m + 2;
    const int om = j > 1 ? m - N : m, op = j < ny ? m + N : m;
#pragma unroll
    for (int i = 0; i < K; ++i) {
      const double2 *pr = reinterpret_cast<const double2 *>(rs.phi + base[c] + i * pl);
      const double2 ym = pr[om], yp = pr[op];
      const double2 fv = f2::ld2x<STREAM>(reinterpret_cast<const double2 *>(rs.f + base[c] + i * pl)[m]);
      const double2 *row = sh + (gc[c] * K + i) * PN;
      const double2 a1 = row[xpad<N>(m1)], b1 = row[xpad<N>(p1)];
      const double a0 = row[xpad<N>(m2)].y, b2 = row[xpad<N>(p2)].x;
      const double2 *zz = z[c] + i;  // planes k-3 .. k+3
      const double2 c0 = zz[3];
      const double lx0 = st0 * c0.x + st1 * (a1.y + c0.y) + st2 * (a1.x + b1.x) + st3 * (a0 + b1.y);
      const double lx1 = st0 * c0.y + st1 * (c0.x + b1.x) + st2 * (a1.y + b1.y) + st3 * (a1.x + b2);
      const double lz0 = st0 * c0.x + st1 * (zz[2].x + zz[4].x) + st2 * (zz[1].x + zz[5].x) + st3 * (zz[0].x + zz[6].x);
      const double lz1 = st0 * c0.y + st1 * (zz[2].y + zz[4].y) + st2 * (zz[1].y + zz[5].y) + st3 * (zz[0].y + zz[6].y);
      const double lap0 = rs.rdx2 * lx0 + rs.rdz2 * lz0 + (am * ym.x + ac * c0.x + ap * yp.x);
      const double lap1 = rs.rdx2 * lx1 + rs.rdz2 * lz1 + (am * ym.y + ac * c0.y + ap * yp.y);
      if (j == 1 && ok[c]) {
        psum += c0.x;
        psum += c0.y;
      }
      r[c][i] = make_double2(fv.x - lap0, fv.y - lap1);
    }
  }
  __syncthreads();  // every thread has read its neighbours
#pragma unroll
  for (int c = 0; c < NC; ++c)
#pragma unroll
    for (int i = 0; i < K; ++i) sh[(gc[c] * K + i) * PN + xpad<N>(mc[c])] = r[c][i];
}

template <int N, typename S, bool STREAM, int SRC>
__global__ void __launch_bounds__(f2_xblock<N>(), (f2_xfwd_min_waves<N, SRC>())) k2_fft_x_fwd(const double *__restrict__ src, S *__restrict__ spec,
                                                    const double2 *__restrict__ tw, const double2 *__restrict__ wx,
                                                    int ny, int nz, int j0, int nj, int pitch, long long rowlen,
                                                    DivSrc dv, ResSrc rs, Geo geo, int tj, int tk) {
  constexpr bool DIV = SRC == kXDiv, COL = SRC == kXResCol, RES = SRC == kXRes || COL, NBR = DIV || RES;
  constexpr int G = f2_threads<N>();
  constexpr int DK = DIV ? f2_div_planes<N>() : 1;
  constexpr int L = DIV ? f2_div_lines<N>() : ((f2_xbase<N>() / G) > 0 ? f2_xbase<N>() / G : 1);
  constexpr int PN = xpadded<N>();
  __shared__ double2 sh[L * PN];
  const int l = threadIdx.x / G, g = threadIdx.x - l * G;
  // lines (j, k) of the planes j0 .. j0+nj-1 (0-based), all k.  Plain rows go
  // j fastest.  DIV reads the uz rows of planes k-1 .. k+2 and the uy rows j,
  // j+1 of each line, RES phi's rows of planes k-3 .. k+3 and j-1, j+1: their
  // lines go in tiles of tj x tk lines (tj | nj, tk | nz; k fastest inside a
  // tile, the tiles k fastest) and runs of two tiles' workgroups go to one XCD
  // (xcd_run), so the neighbouring lines that re-read a row, in j or in k, do
  // so through the same L2.
  const unsigned nzp = DK > 1 ? (nz + DK - 1) / DK * DK : nz;  // whole groups of planes
  const unsigned nlines = (unsigned)nj * nzp;
  const int tt = tj * tk;
  const unsigned wb = NBR ? (unsigned)xcd_run((int)blockIdx.x, (int)gridDim.x, tt >= L ? 2 * tt / L : 1) : blockIdx.x;
  const unsigned q = wb * L + l;
  const LineAt at = line_at<NBR>(l < L && q < nlines ? q : 0, nj, nzp, tj, tk);
  const bool live = l < L && q < nlines && (DK == 1 || at.k < nz);
  const long long jl = j0 + at.j, k = at.k;
  const long long sq = jl + (long long)ny * k;  // spectral row S[k][jl]
  const double2 *row = reinterpret_cast<const double2 *>(src + rowlen * (jl + 1 + (long long)(ny + 2) * k));
  double2 *ls = sh + (l < L ? l : 0) * PN;
  double dmax = 0.0;
  auto load_div = [&](int m) { return div_pair(dv, geo, N, ny, nz, rowlen, jl, k, m, dmax); };
  double psum = 0.0;
  auto load_res = [&](int m) {
    // the pair of points (2m, 2m+1) of row j = jl + 1, plane k
    constexpr double st0 = -1460.0 / 576.0, st1 = 783.0 / 576.0, st2 = -54.0 / 576.0, st3 = 1.0 / 576.0;
    const long long rj = rowlen * (jl + 1 + (long long)(ny + 2) * k);
    const double2 *pr = reinterpret_cast<const double2 *>(rs.phi + rj);
    double2 p[5];  // pairs m-2 .. m+2: points 2m-4 .. 2m+5
#pragma unroll
    for (int s = 0; s < 5; ++s) {
      int mm = m + s - 2;
      mm = mm < 0 ? mm + N : (mm >= N ? mm - N : mm);
      p[s] = pr[mm];
    }
    const long long pl = rowlen * (ny + 2);
    double2 z[7];
#pragma unroll
    for (int s = 0; s < 7; ++s) {
      long long kk = k - 3 + s;
      kk = kk < 0 ? kk + nz : (kk >= nz ? kk - nz : kk);
      z[s] = reinterpret_cast<const double2 *>(rs.phi + rj + (kk - k) * pl)[m];
    }
    const int j = (int)jl + 1;
    const double2 c0 = p[2];
    const double2 ym = j > 1 ? pr[m - N] : c0, yp = j < ny ? pr[m + N] : c0;
    const double2 fv = reinterpret_cast<const double2 *>(rs.f + rj)[m];
    const double am = geo.met[M_AM2PH * geo.nyh + j], ac = geo.met[M_AC2PH * geo.nyh + j],
                 ap = geo.met[M_AP2PH * geo.nyh + j];
    const double lx0 = st0 * c0.x + st1 * (p[1].y + c0.y) + st2 * (p[1].x + p[3].x) + st3 * (p[0].y + p[3].y);
    const double lx1 = st0 * c0.y + st1 * (c0.x + p[3].x) + st2 * (p[1].y + p[3].y) + st3 * (p[1].x + p[4].x);
    const double lz0 = st0 * c0.x + st1 * (z[2].x + z[4].x) + st2 * (z[1].x + z[5].x) + st3 * (z[0].x + z[6].x);
    const double lz1 = st0 * c0.y + st1 * (z[2].y + z[4].y) + st2 * (z[1].y + z[5].y) + st3 * (z[0].y + z[6].y);
    const double lap0 = rs.rdx2 * lx0 + rs.rdz2 * lz0 + (am * ym.x + ac * c0.x + ap * yp.x);
    const double lap1 = rs.rdx2 * lx1 + rs.rdz2 * lz1 + (am * ym.y + ac * c0.y + ap * yp.y);
    if (j == 1) {
      psum += c0.x;
      psum += c0.y;
    }
    return make_double2(fv.x - lap0, fv.y - lap1);
  };
  auto load0 = [&](int m) {
    if (!live) return make_double2(0.0, 0.0);
    if constexpr (DIV) return load_div(m);
    else if constexpr (RES) return load_res(m);
    else return f2::ld2x<STREAM>(row[m]);
  };
  auto lds = [&](int m) -> double2 & { return ls[xpad<N>(m)]; };
  auto store_lds = [&](int m, double2 v) { ls[xpad<N>(m)] = v; };
  if constexpr (COL) {
    res_columns<N, f2_res_lines<N>(), STREAM>(sh, rs, geo, ny, nz, rowlen, j0, wb * L, nlines, tj, tk, psum);
    __syncthreads();
    f2::run_fft<N, G, false, true>(g, tw, lds, lds, store_lds);
  } else if constexpr (DK > 1) {
    div_columns<DK>(dv, geo, N, ny, nz, (int)nzp, rowlen, j0, nlines, tj, tk, wb * L, L, f2_xblock<N>(),
                    [&](int line, int m) -> double2 & { return sh[line * PN + xpad<N>(m)]; }, dmax);
    __syncthreads();
    f2::run_fft<N, G, false, true>(g, tw, lds, lds, store_lds);
  } else {
    f2::run_fft<N, G, false>(g, tw, load0, lds, store_lds);
  }
  __syncthreads();
  if (live) x_untangle_store<N, G, STREAM>(g, ls, wx, spec + sq * pitch, pitch);
  if constexpr (DIV) {
    // in the FFT's LDS once its reads are done
    const double dm = block_max_tree(dmax, reinterpret_cast<double *>(sh));
    if (threadIdx.x == 0) dv.part[blockIdx.x] = dm;
  }
  if constexpr (RES) {
    // fixed-order tree over the workgroup, in the FFT's LDS once its reads are done
    double *red = reinterpret_cast<double *>(sh);
    __syncthreads();
    red[threadIdx.x] = psum;
    __syncthreads();
    for (int n = blockDim.x; n > 1;) {
      const int h = (n + 1) / 2;
      if ((int)threadIdx.x < n - h) red[threadIdx.x] += red[threadIdx.x + h];
      __syncthreads();
      n = h;
    }
    if (threadIdx.x == 0) rs.psum[blockIdx.x] = red[0];
  }
}

// ---- x inverse: half spectra -> real rows times scale ----------------------
// ACC: add the result to dst (a correction) instead of storing it, minus the
// device scalar *shift (the mean the correction removes).  ghost: the rows
// j = 1 and j = ny also go to the Neumann ghost rows j = 0 and j = ny+1
// (SetBC_and_UpdateHalo_pr, src/m_BC_and_Halo.f90:115-120).

template <int N, typename S, bool ACC, bool STREAM>
__global__ void __launch_bounds__(f2_xblock<N>(), f2_x_min_waves<N>())
    k2_fft_x_inv(const S *__restrict__ spec, double *__restrict__ dst,
                                                    const double2 *__restrict__ tw, const double2 *__restrict__ wx,
                                                    int ny, int nz, int j0, int nj, int pitch, long long rowlen,
                                                    double scale, const double *__restrict__ shift, int ghost) {
  constexpr int G = f2_threads<N>();
  constexpr int L = (f2_xbase<N>() / G) > 0 ? f2_xbase<N>() / G : 1;
  constexpr int PN = xpadded<N>();
  __shared__ double2 sh[L * PN];
  const int l = threadIdx.x / G, g = threadIdx.x - l * G;
  const unsigned q = blockIdx.x * L + l;
  const bool live = l < L && q < (unsigned)nj * nz;
  const LineAt at = line_at<false>(live ? q : 0, nj, nz, 1, 1);
  const long long jl = j0 + at.j, k = at.k;
  const S *in = spec + (jl + (long long)ny * k) * pitch;
  double2 *ls = sh + (l < L ? l : 0) * PN;
  // The re-tangle of element m needs X_m and X_{N-m}: the line's N+1 values
  // go through LDS once (coalesced) instead of being fetched twice.  All of a
  // thread's loads are issued before the first LDS write (lines past the end
  // read line 0 and store nothing; indices past N repeat element N, so
  // every thread that reaches it writes the same value).
  constexpr int NT = N / G + 1;
  double2 pre[NT];
#pragma unroll
  for (int t = 0; t < NT; ++t) pre[t] = f2::ld2x<STREAM>(in[min(g + t * G, N)]);
#pragma unroll
  for (int t = 0; t < NT; ++t) ls[xpad<N>(min(g + t * G, N))] = pre[t];
  __syncthreads();
  auto load0 = [&](int m) { return x_retangle<N>(ls, wx, m); };
  auto lds = [&](int m) -> double2 & { return ls[xpad<N>(m)]; };
  double2 *row = reinterpret_cast<double2 *>(dst + rowlen * (jl + 1 + (long long)(ny + 2) * k));
  // the ghost row this line also fills (or none)
  double2 *grow = nullptr;
  if (ghost && jl == 0) grow = reinterpret_cast<double2 *>(dst + rowlen * ((long long)(ny + 2) * k));
  if (ghost && jl == ny - 1) grow = reinterpret_cast<double2 *>(dst + rowlen * (ny + 1 + (long long)(ny + 2) * k));
  const double sh0 = ACC ? shift[0] : 0.0;
  auto store_out = [&](int m, double2 v) {
    if (!live) return;
    double2 x;
    if (ACC) {
      const double2 o = f2::ld2x<STREAM>(row[m]);
      x = make_double2(o.x + v.x * scale - sh0, o.y + v.y * scale - sh0);
    } else {
      x = make_double2(v.x * scale, v.y * scale);
    }
    f2::st2x<STREAM>(row[m], x);
    if (grow) f2::st2x<STREAM>(grow[m], x);
  };
  f2::run_fft<N, G, true, true>(g, tw, load0, lds, store_out);
}

// ---- z pass: T columns x N rows, thread id = g * T + col ----------------
// 1-D grid of ntile * nj workgroups: column tile and plane from the
// XCD-grouped index, so that the tiles sharing a 128-byte row segment (narrow
// tiles of the long lengths) are read and written through one L2.
template <int N, int T, bool INV, typename S>
__global__ void __launch_bounds__(f2_threads<N>() * T) k2_fft_z(S *__restrict__ spec, const double2 *__restrict__ tw, int ny,
                                                 int pitch, int j0, int ntile) {
  constexpr int G = f2_threads<N>();
  constexpr int GRP = (int)(128 / (T * sizeof(S))) > 1 ? (int)(128 / (T * sizeof(S))) : 1;
  __shared__ double2 sh[N * T];
  const int col = threadIdx.x % T, g = threadIdx.x / T;
  const long long zs = (long long)pitch * ny;
  const int w = xcd_group<GRP>((int)blockIdx.x, (int)gridDim.x);
  const int tile = w % ntile, jj = w / ntile;
  S *base = spec + (long long)(j0 + jj) * pitch + (long long)tile * T + col;
  auto load0 = [&](int m) { return f2::ld2(base[m * zs]); };
  auto lds = [&](int m) -> double2 & { return sh[m * T + col]; };
  auto store_out = [&](int m, double2 v) { f2::st2(base[m * zs], v); };
  f2::run_fft<N, G, INV>(g, tw, load0, lds, store_out);
}

// ---- persistent passes with a register prefetch of the next work item ------
// The long lengths keep one workgroup per CU (their lines fill 83-90 KB of
// LDS), so a one-shot workgroup idles through the HBM latency of its own
// loads and the CU has no other workgroup to switch to.  These kernels run
// one or a few workgroups per CU over the work items (line groups, or z
// column tiles) in strides of the grid; each issues the global loads of its
// next item -- the inputs of stage 0, straight into the registers stage 0
// of the current item has just consumed -- before the remaining stages, so
// those loads are in flight during the LDS stages.  The barriers wait on LDS traffic only (s_waitcnt lgkmcnt), not
// on the outstanding global loads.  Same arithmetic as the one-shot kernels.

template <int N, typename S, bool STREAM>
__global__ void __launch_bounds__(f2_xblock<N>()) k2p_fft_x_fwd(const double *__restrict__ src, S *__restrict__ spec,
                                                     const double2 *__restrict__ tw, const double2 *__restrict__ wx,
                                                     int ny, int nz, int j0, int nj, int pitch, long long rowlen) {
  constexpr int G = f2_threads<N>();
  constexpr int L = (f2_xbase<N>() / G) > 0 ? f2_xbase<N>() / G : 1;
  constexpr int PN = xpadded<N>();
  constexpr int R0 = f2::make_plan(N).r[0];
  constexpr int NB0 = N / R0;
  constexpr int BPT0 = f2::stage_bpt<N, 0, G>();
  __shared__ double2 sh[L * PN];
  const int l = threadIdx.x / G, g = threadIdx.x - l * G;
  const unsigned nlines = (unsigned)nj * nz;
  const long long ngroups = (nlines + L - 1) / L;
  double2 *ls = sh + l * PN;
  // line l of group grp: rows j fastest; sq = its spectral row
  auto line = [&](long long grp, bool &live, long long &sq) {
    const unsigned q = (unsigned)grp * L + l;
    live = q < nlines;
    const LineAt at = line_at<false>(live ? q : 0, nj, nz, 1, 1);
    const long long jl = j0 + at.j, k = at.k;
    sq = jl + (long long)ny * k;
    return reinterpret_cast<const double2 *>(src + rowlen * (jl + 1 + (long long)(ny + 2) * k));
  };
  auto fetch = [&](long long grp, f2::StageRegs<N, 0, G> &v) {
    bool live;
    long long sq;
    const double2 *row = line(grp, live, sq);
#pragma unroll
    for (int i = 0; i < BPT0; ++i) {
      const int b = g + i * G;
      if (BPT0 * G == NB0 || b < NB0) {
#pragma unroll
        for (int r = 0; r < R0; ++r) v[i][r] = live ? f2::ld2x<STREAM>(row[b + r * NB0]) : make_double2(0.0, 0.0);
      }
    }
  };
  auto lds = [&](int m) -> double2 & { return ls[xpad<N>(m)]; };
  auto store_lds = [&](int m, double2 v) { ls[xpad<N>(m)] = v; };
  f2::StageRegs<N, 0, G> v;
  long long grp = blockIdx.x;
  if (grp >= ngroups) return;
  fetch(grp, v);
  for (; grp < ngroups; grp += gridDim.x) {
    // the lane index through an empty asm: the per-stage LDS addresses are
    // recomputed in each iteration, as in the one-shot kernel, rather than
    // hoisted out of the loop into registers
    int gi = g;
    asm volatile("" : "+v"(gi));
    // the stage twiddles, reloaded per item (cache hits) rather than held
    // across the loop
    double2 W[7][4];
    f2::load_twiddles<N, G, false>(gi, tw, W);
    // stage 0 consumes the registers; the next group's loads then go into
    // them (the last group re-reads its own: no branch around the loads, and
    // the values are discarded).  The scheduling barrier keeps those loads
    // after stage 0, so the two sets of registers are never live together.
    f2::stage_exec<N, 0, G, false>(gi, W[0], v, store_lds);
    __builtin_amdgcn_sched_barrier(0);
    const long long gn = grp + gridDim.x < ngroups ? grp + gridDim.x : grp;
    fetch(gn, v);
    __syncthreads();
    f2::run_rest<N, G, false>(gi, W, lds, store_lds);
    __syncthreads();
    bool live;
    long long sq;
    (void)line(grp, live, sq);
    if (live) x_untangle_store<N, G, STREAM>(gi, ls, wx, spec + sq * pitch, pitch);
    __syncthreads();
  }
}

template <int N, typename S, bool ACC, bool STREAM>
__global__ void __launch_bounds__(f2_xblock<N>()) k2p_fft_x_inv(const S *__restrict__ spec, double *__restrict__ dst,
                                                     const double2 *__restrict__ tw, const double2 *__restrict__ wx,
                                                     int ny, int nz, int j0, int nj, int pitch, long long rowlen,
                                                     double scale, const double *__restrict__ shift, int ghost) {
  constexpr int G = f2_threads<N>();
  constexpr int L = (f2_xbase<N>() / G) > 0 ? f2_xbase<N>() / G : 1;
  constexpr int PN = xpadded<N>();
  constexpr int NT = N / G + 1;
  __shared__ double2 sh[L * PN];
  const int l = threadIdx.x / G, g = threadIdx.x - l * G;
  const unsigned nlines = (unsigned)nj * nz;
  const long long ngroups = (nlines + L - 1) / L;
  double2 *ls = sh + l * PN;
  const double sh0 = ACC ? shift[0] : 0.0;
  auto coords = [&](long long grp, bool &live, long long &jl, long long &k) {
    const unsigned q = (unsigned)grp * L + l;
    live = q < nlines;
    const LineAt at = line_at<false>(live ? q : 0, nj, nz, 1, 1);
    jl = j0 + at.j;
    k = at.k;
  };
  // the line's N+1 spectral values (indices past N repeat element N)
  auto fetch = [&](long long grp, double2 (&v)[NT]) {
    bool live;
    long long jl, k;
    coords(grp, live, jl, k);
    const S *in = spec + (jl + (long long)ny * k) * pitch;
#pragma unroll
    for (int t = 0; t < NT; ++t) v[t] = f2::ld2x<STREAM>(in[min(g + t * G, N)]);
  };
  auto lds = [&](int m) -> double2 & { return ls[xpad<N>(m)]; };
  double2 v[NT];
  long long grp = blockIdx.x;
  if (grp >= ngroups) return;
  fetch(grp, v);
  for (; grp < ngroups; grp += gridDim.x) {
    int gi = g;  // recomputed addresses and twiddles per iteration, as in the forward pass
    asm volatile("" : "+v"(gi));
    double2 W[7][4];
    f2::load_twiddles<N, G, true>(gi, tw, W);
#pragma unroll
    for (int t = 0; t < NT; ++t) ls[xpad<N>(min(gi + t * G, N))] = v[t];
    // the registers are free: the next group's loads go into them
    __builtin_amdgcn_sched_barrier(0);
    const long long gn = grp + gridDim.x < ngroups ? grp + gridDim.x : grp;
    fetch(gn, v);
    __syncthreads();
    bool live;
    long long jl, k;
    coords(grp, live, jl, k);
    double2 *row = reinterpret_cast<double2 *>(dst + rowlen * (jl + 1 + (long long)(ny + 2) * k));
    double2 *grow = nullptr;
    if (ghost && jl == 0) grow = reinterpret_cast<double2 *>(dst + rowlen * ((long long)(ny + 2) * k));
    if (ghost && jl == ny - 1) grow = reinterpret_cast<double2 *>(dst + rowlen * (ny + 1 + (long long)(ny + 2) * k));
    auto load0 = [&](int m) { return x_retangle<N>(ls, wx, m); };
    auto store_out = [&](int m, double2 v) {
      if (!live) return;
      double2 x;
      if (ACC) {
        const double2 o = f2::ld2x<STREAM>(row[m]);
        x = make_double2(o.x + v.x * scale - sh0, o.y + v.y * scale - sh0);
      } else {
        x = make_double2(v.x * scale, v.y * scale);
      }
      f2::st2x<STREAM>(row[m], x);
      if (grow) f2::st2x<STREAM>(grow[m], x);
    };
    f2::run_fft_w<N, G, true, true>(gi, W, load0, lds, store_out);
    __syncthreads();
  }
}

// z pass over nitems = ntile * nj column tiles (XCD-grouped as the one-shot
// kernel, so the tiles that share a 128-byte row segment are in flight on
// one XCD together)
template <int N, int T, bool INV, typename S>
__global__ void __launch_bounds__(f2_threads<N>() * T) k2p_fft_z(S *__restrict__ spec, const double2 *__restrict__ tw,
                                                  int ny, int pitch, int j0, int ntile, int nitems) {
  constexpr int G = f2_threads<N>();
  constexpr int GRP = (int)(128 / (T * sizeof(S))) > 1 ? (int)(128 / (T * sizeof(S))) : 1;
  constexpr int R0 = f2::make_plan(N).r[0];
  constexpr int NB0 = N / R0;
  constexpr int BPT0 = f2::stage_bpt<N, 0, G>();
  __shared__ double2 sh[N * T];
  const int col = threadIdx.x % T, g = threadIdx.x / T;
  const long long zs = (long long)pitch * ny;
  auto base_of = [&](int item) {
    const int w = xcd_group<GRP>(item, nitems);
    const int tile = w % ntile, jj = w / ntile;
    return spec + (long long)(j0 + jj) * pitch + (long long)tile * T + col;
  };
  auto fetch = [&](int item, f2::StageRegs<N, 0, G> &v) {
    const S *base = base_of(item);
#pragma unroll
    for (int i = 0; i < BPT0; ++i) {
      const int b = g + i * G;
      if (BPT0 * G == NB0 || b < NB0) {
#pragma unroll
        for (int r = 0; r < R0; ++r) v[i][r] = f2::ld2(base[(long long)(b + r * NB0) * zs]);
      }
    }
  };
  f2::StageRegs<N, 0, G> v;
  int item = blockIdx.x;
  if (item >= nitems) return;
  fetch(item, v);
  for (; item < nitems; item += gridDim.x) {
    // lane indices through an empty asm: addresses recomputed per iteration
    int tid = (int)threadIdx.x;
    asm volatile("" : "+v"(tid));
    const int ci = tid % T, gi = tid / T;
    double2 W[7][4];
    f2::load_twiddles<N, G, INV>(gi, tw, W);
    auto lds = [&](int m) -> double2 & { return sh[m * T + ci]; };
    auto store_lds = [&](int m, double2 x) { sh[m * T + ci] = x; };
    f2::stage_exec<N, 0, G, INV>(gi, W[0], v, store_lds);
    __builtin_amdgcn_sched_barrier(0);
    const int in = item + (int)gridDim.x < nitems ? item + (int)gridDim.x : item;
    fetch(in, v);
    S *base = base_of(item);
    auto store_out = [&](int m, double2 x) { f2::st2(base[(long long)m * zs], x); };
    __syncthreads();
    f2::run_rest<N, G, INV>(gi, W, lds, store_out);
    __syncthreads();
  }
}

// ---- dispatch ----------------------------------------------------------------
// lengths with persistent forms: the x lengths of the 1024-, 4608- and
// 9216-point rows, the z length 1400 with its 2- and 4-column tiles.  The
// shorter z lengths run faster one-shot: at 1024x256x512 the 8-column pass
// took 0.416 ms against 0.438 (16 columns, 44 bytes of scratch per lane at the
// 128 VGPRs of a 1024-thread workgroup, 1.34x the read bytes) and 0.456 (8
// columns) persistent; at 4608x140x700 1.77 ms against 1.80-1.82 (8 columns,
// 28 bytes of scratch per lane) and 2.18 (4 columns).
constexpr bool has_px(int n) { return n == 512 || n == 2304 || n == 4608; }
constexpr bool has_pz(int n, int t) { return n == 1400 && (t == 2 || t == 4); }

// workgroups of a persistent kernel resident per CU (at least one)
template <class K>
static int resident_blocks(K kernel, int threads) {
  int nb = 0;
  if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&nb, kernel, threads, 0) != hipSuccess || nb < 1) {
    (void)hipGetLastError();
    nb = 1;
  }
  return nb;
}

static unsigned persistent_grid(const ptc_ctx *c, int per_cu, long long items) {
  return (unsigned)std::max<long long>(1, std::min<long long>(items, (long long)per_cu * std::max(1, c->n_cu)));
}

template <int N, typename S, bool STREAM>
static void px_fwd_launch(ptc_ctx *c, const double *src, S *spec, int j0, int nj) {
  constexpr int G = f2_threads<N>();
  constexpr int L = (f2_xbase<N>() / G) > 0 ? f2_xbase<N>() / G : 1;
  static const int per_cu = resident_blocks(k2p_fft_x_fwd<N, S, STREAM>, L * G);
  const long long groups = ((long long)nj * c->nz + L - 1) / L;
  hipLaunchKernelGGL((k2p_fft_x_fwd<N, S, STREAM>), dim3(persistent_grid(c, per_cu, groups)), dim3(L * G), 0,
                     c->stream, src, spec, c->pp.fx.tw, c->pp.d_wx, c->ny, c->nz, j0, nj, c->pp.pitch,
                     (long long)c->nx);
}

template <int N, typename S, bool ACC, bool STREAM>
static void px_inv_launch(ptc_ctx *c, const S *spec, double *dst, double scale, int j0, int nj, bool ghost) {
  constexpr int G = f2_threads<N>();
  constexpr int L = (f2_xbase<N>() / G) > 0 ? f2_xbase<N>() / G : 1;
  static const int per_cu = resident_blocks(k2p_fft_x_inv<N, S, ACC, STREAM>, L * G);
  const long long groups = ((long long)nj * c->nz + L - 1) / L;
  hipLaunchKernelGGL((k2p_fft_x_inv<N, S, ACC, STREAM>), dim3(persistent_grid(c, per_cu, groups)), dim3(L * G), 0,
                     c->stream, spec, dst, c->pp.fx.tw, c->pp.d_wx, c->ny, c->nz, j0, nj, c->pp.pitch,
                     (long long)c->nx, scale, c->d_scal + kSlotPinShift, ghost ? 1 : 0);
}

template <int N, int T, bool INV, typename S>
static void pz_launch(ptc_ctx *c, S *spec, int j0, int nj) {
  constexpr int G = f2_threads<N>();
  static const int per_cu = resident_blocks(k2p_fft_z<N, T, INV, S>, G * T);
  const int ntile = c->pp.pitch / T;
  const int nitems = ntile * nj;
  hipLaunchKernelGGL((k2p_fft_z<N, T, INV, S>), dim3(persistent_grid(c, per_cu, nitems)), dim3(G * T), 0, c->stream,
                     spec, c->pp.fz.tw, c->ny, c->pp.pitch, j0, ntile, nitems);
}

template <int N>
static long long x_fwd_blocks(long long nlines) {
  constexpr int G = f2_threads<N>();
  constexpr int L = (f2_xbase<N>() / G) > 0 ? f2_xbase<N>() / G : 1;
  return (nlines + L - 1) / L;
}

// workgroups of the divergence-forming pass
template <int N>
static long long x_div_blocks(int nj, int nz) {
  constexpr int K = f2_div_planes<N>(), L = f2_div_lines<N>();
  return ((long long)nj * ((nz + K - 1) / K * K) + L - 1) / L;
}

template <int N, typename S, bool STREAM, int SRC>
static void x_fwd_launch(ptc_ctx *c, const double *src, S *spec, int j0, int nj, const DivSrc &dv,
                         const ResSrc &rs = ResSrc{}) {
  constexpr int G = f2_threads<N>();
  constexpr int L = (f2_xbase<N>() / G) > 0 ? f2_xbase<N>() / G : 1;
  constexpr int DK = SRC == kXDiv ? f2_div_planes<N>() : 1;
  const unsigned nblk = (unsigned)(SRC == kXDiv ? x_div_blocks<N>(nj, c->nz) : x_fwd_blocks<N>((long long)nj * c->nz));
  int tj, tk;
  line_tile(nj, (c->nz + DK - 1) / DK * DK, &tj, &tk);
  hipLaunchKernelGGL((k2_fft_x_fwd<N, S, STREAM, SRC>), dim3(nblk), dim3(DK > 1 ? f2_xblock<N>() : L * G), 0, c->stream, src, spec,
                     c->pp.fx.tw, c->pp.d_wx, c->ny, c->nz, j0, nj, c->pp.pitch, (long long)c->nx, dv, rs, c->geo,
                     tj, tk);
}

// the residual by columns where the length has the form and the tiles of
// lines hold whole groups of its planes, else pair by pair
template <int N, bool STREAM>
static void x_res_launch(ptc_ctx *c, float2 *spec, int j0, int nj, const ResSrc &res) {
  constexpr int K = f2_res_lines<N>();
  if constexpr (K > 0) {
    int tj, tk;
    line_tile(nj, c->nz, &tj, &tk);
    if (tk % K == 0) {
      x_fwd_launch<N, float2, STREAM, kXResCol>(c, nullptr, spec, j0, nj, DivSrc{}, res);
      return;
    }
  }
  x_fwd_launch<N, float2, STREAM, kXRes>(c, nullptr, spec, j0, nj, DivSrc{}, res);
}

template <int N>
static int x_fwd_t(ptc_ctx *c, const double *src, void *spec, int j0, int nj, bool f64, const DivSrc *div,
                   const ResSrc *res) {
  const bool f32 = !f64 && c->pp.prec == PTC_PREC_FP32_REFINE;
  const DivSrc none{};
  if (div) {
    PTC_CHECK(!f32, PTC_E_STATE, "the divergence-forming x pass needs FP64 spectra");
    if (c->pp.stream) x_fwd_launch<N, double2, true, kXDiv>(c, src, (double2 *)spec, j0, nj, *div);
    else x_fwd_launch<N, double2, false, kXDiv>(c, src, (double2 *)spec, j0, nj, *div);
  } else if (res) {
    // the one-shot kernel forms the residual, whatever the plan's x form
    PTC_CHECK(f32, PTC_E_STATE, "the residual-forming x pass belongs to the FP32-storage refinement");
    if (c->pp.stream) x_res_launch<N, true>(c, (float2 *)spec, j0, nj, *res);
    else x_res_launch<N, false>(c, (float2 *)spec, j0, nj, *res);
  } else if (c->pp.persist_x) {
    if constexpr (has_px(N)) {
      if (f32 && c->pp.stream) px_fwd_launch<N, float2, true>(c, src, (float2 *)spec, j0, nj);
      else if (f32) px_fwd_launch<N, float2, false>(c, src, (float2 *)spec, j0, nj);
      else if (c->pp.stream) px_fwd_launch<N, double2, true>(c, src, (double2 *)spec, j0, nj);
      else px_fwd_launch<N, double2, false>(c, src, (double2 *)spec, j0, nj);
    } else {
      set_error("no persistent x pass for this length");
      return PTC_E_UNSUPPORTED;
    }
  } else if (f32 && c->pp.stream) {
    x_fwd_launch<N, float2, true, kXPlain>(c, src, (float2 *)spec, j0, nj, none);
  } else if (f32) {
    x_fwd_launch<N, float2, false, kXPlain>(c, src, (float2 *)spec, j0, nj, none);
  } else if (c->pp.stream) {
    x_fwd_launch<N, double2, true, kXPlain>(c, src, (double2 *)spec, j0, nj, none);
  } else {
    x_fwd_launch<N, double2, false, kXPlain>(c, src, (double2 *)spec, j0, nj, none);
  }
  PTC_HIP(hipGetLastError());
  return PTC_OK;
}

template <int N, typename S, bool ACC, bool STREAM>
static void x_inv_launch(ptc_ctx *c, const S *spec, double *dst, double scale, int j0, int nj, bool ghost) {
  constexpr int G = f2_threads<N>();
  constexpr int L = (f2_xbase<N>() / G) > 0 ? f2_xbase<N>() / G : 1;
  const long long nlines = (long long)nj * c->nz;
  const unsigned nblk = (unsigned)((nlines + L - 1) / L);
  hipLaunchKernelGGL((k2_fft_x_inv<N, S, ACC, STREAM>), dim3(nblk), dim3(L * G), 0, c->stream, spec, dst,
                     c->pp.fx.tw, c->pp.d_wx, c->ny, c->nz, j0, nj, c->pp.pitch, (long long)c->nx, scale,
                     c->d_scal + kSlotPinShift, ghost ? 1 : 0);
}

template <int N>
static int x_inv_t(ptc_ctx *c, const void *spec, double *dst, double scale, int j0, int nj, bool acc, bool ghost) {
  const bool f32 = c->pp.prec == PTC_PREC_FP32_REFINE, st = c->pp.stream;
  const float2 *s4 = (const float2 *)spec;
  const double2 *s8 = (const double2 *)spec;
  if (c->pp.persist_x) {
    if constexpr (has_px(N)) {
      if (f32) {
        if (acc && st) px_inv_launch<N, float2, true, true>(c, s4, dst, scale, j0, nj, ghost);
        else if (acc) px_inv_launch<N, float2, true, false>(c, s4, dst, scale, j0, nj, ghost);
        else if (st) px_inv_launch<N, float2, false, true>(c, s4, dst, scale, j0, nj, ghost);
        else px_inv_launch<N, float2, false, false>(c, s4, dst, scale, j0, nj, ghost);
      } else {
        PTC_CHECK(!acc, PTC_E_STATE, "accumulating x-inverse with FP64 spectra");
        if (st) px_inv_launch<N, double2, false, true>(c, s8, dst, scale, j0, nj, ghost);
        else px_inv_launch<N, double2, false, false>(c, s8, dst, scale, j0, nj, ghost);
      }
      PTC_HIP(hipGetLastError());
      return PTC_OK;
    } else {
      set_error("no persistent x pass for this length");
      return PTC_E_UNSUPPORTED;
    }
  }
  if (f32) {
    if (acc && st) x_inv_launch<N, float2, true, true>(c, s4, dst, scale, j0, nj, ghost);
    else if (acc) x_inv_launch<N, float2, true, false>(c, s4, dst, scale, j0, nj, ghost);
    else if (st) x_inv_launch<N, float2, false, true>(c, s4, dst, scale, j0, nj, ghost);
    else x_inv_launch<N, float2, false, false>(c, s4, dst, scale, j0, nj, ghost);
  } else {
    // the accumulating form belongs to the FP32-storage refinement only
    PTC_CHECK(!acc, PTC_E_STATE, "accumulating x-inverse with FP64 spectra");
    if (st) x_inv_launch<N, double2, false, true>(c, s8, dst, scale, j0, nj, ghost);
    else x_inv_launch<N, double2, false, false>(c, s8, dst, scale, j0, nj, ghost);
  }
  PTC_HIP(hipGetLastError());
  return PTC_OK;
}

template <int N, int T>
static int z_t(ptc_ctx *c, void *spec, bool inverse, int j0, int nj, bool f64) {
  constexpr int G = f2_threads<N>();
  const int ntile = c->pp.pitch / T;
  dim3 grid((unsigned)(ntile * nj));
  const auto *tw = c->pp.fz.tw;
  const int ny = c->ny, pitch = c->pp.pitch;
  if (c->pp.persist_z) {
    if constexpr (has_pz(N, T)) {
      if (!f64 && c->pp.prec == PTC_PREC_FP32_REFINE) {
        if (inverse) pz_launch<N, T, true, float2>(c, (float2 *)spec, j0, nj);
        else pz_launch<N, T, false, float2>(c, (float2 *)spec, j0, nj);
      } else {
        if (inverse) pz_launch<N, T, true, double2>(c, (double2 *)spec, j0, nj);
        else pz_launch<N, T, false, double2>(c, (double2 *)spec, j0, nj);
      }
      PTC_HIP(hipGetLastError());
      return PTC_OK;
    } else {
      set_error("no persistent z pass for this length and tile");
      return PTC_E_UNSUPPORTED;
    }
  }
  if (!f64 && c->pp.prec == PTC_PREC_FP32_REFINE) {
    if (inverse)
      hipLaunchKernelGGL((k2_fft_z<N, T, true, float2>), grid, dim3(G * T), 0, c->stream, (float2 *)spec, tw, ny, pitch,
                         j0, ntile);
    else
      hipLaunchKernelGGL((k2_fft_z<N, T, false, float2>), grid, dim3(G * T), 0, c->stream, (float2 *)spec, tw, ny,
                         pitch, j0, ntile);
  } else {
    if (inverse)
      hipLaunchKernelGGL((k2_fft_z<N, T, true, double2>), grid, dim3(G * T), 0, c->stream, (double2 *)spec, tw, ny,
                         pitch, j0, ntile);
    else
      hipLaunchKernelGGL((k2_fft_z<N, T, false, double2>), grid, dim3(G * T), 0, c->stream, (double2 *)spec, tw, ny,
                         pitch, j0, ntile);
  }
  PTC_HIP(hipGetLastError());
  return PTC_OK;
}

// x lengths h = nx/2 with a specialised kernel
// (2304 and 4608: the 4608- and 9216-point rows of the largest cases; their
// lines take 41 KB and 83 KB of LDS, which gfx950's 160 KB allows)
#define PTC_X_SIZES(X) X(8) X(16) X(32) X(48) X(64) X(96) X(128) X(256) X(512) X(768) X(2304) X(4608)

bool fft2_has_px(int h) { return has_px(h); }
bool fft2_has_pz(int nz, int tile) { return has_pz(nz, tile); }

bool fft2_has_x(int h) {
#define PTC_CASE(N) if (h == N) return true;
  PTC_X_SIZES(PTC_CASE)
#undef PTC_CASE
  return false;
}

int fft2_x_fwd(ptc_ctx *c, const double *src, void *spec, int j0, int nj, bool f64, const DivSrc *div,
               const ResSrc *res) {
  switch (c->pp.h) {
#define PTC_CASE(N) case N: return x_fwd_t<N>(c, src, spec, j0, nj, f64, div, res);
    PTC_X_SIZES(PTC_CASE)
#undef PTC_CASE
    default: return PTC_E_UNSUPPORTED;
  }
}

long long fft2_x_fwd_blocks(const ptc_ctx *c, int nj) {
  switch (c->pp.h) {
#define PTC_CASE(N) case N: return x_fwd_blocks<N>((long long)nj * c->nz);
    PTC_X_SIZES(PTC_CASE)
#undef PTC_CASE
    default: return 0;
  }
}

long long fft2_x_div_blocks(const ptc_ctx *c, int nj) {
  switch (c->pp.h) {
#define PTC_CASE(N) case N: return x_div_blocks<N>(nj, c->nz);
    PTC_X_SIZES(PTC_CASE)
#undef PTC_CASE
    default: return 0;
  }
}

int fft2_x_inv(ptc_ctx *c, const void *spec, double *dst, double scale, int j0, int nj, bool acc, bool ghost) {
  switch (c->pp.h) {
#define PTC_CASE(N) case N: return x_inv_t<N>(c, spec, dst, scale, j0, nj, acc, ghost);
    PTC_X_SIZES(PTC_CASE)
#undef PTC_CASE
    default: return PTC_E_UNSUPPORTED;
  }
}

// z lengths with a specialised kernel and their column tile (<= 64 KB LDS,
// <= 512 threads): the default tile of each length
#define PTC_Z_SIZES(Z) \
  Z(16, 16) Z(32, 16) Z(64, 16) Z(96, 16) Z(128, 16) Z(192, 16) Z(256, 16) Z(512, 8) Z(700, 4) Z(1400, 2)
// wider alternatives for the autotuner: 256-byte row segments, one 1024-thread
// workgroup of 128 KB LDS per CU; for the long lengths twice the default
// tile, one workgroup of 90 KB LDS per CU
#define PTC_Z_WIDE(Z) Z(256, 32) Z(512, 16) Z(700, 8) Z(1400, 4)

// req = 0: the default tile; else that tile if compiled for nz
bool fft2_has_z(int nz, int req, int *tile) {
#define PTC_CASE(N, T) \
  if (nz == N && (req == 0 || req == T)) { *tile = T; return true; }
  PTC_Z_SIZES(PTC_CASE)
  PTC_Z_WIDE(PTC_CASE)
#undef PTC_CASE
  return false;
}

int fft2_z(ptc_ctx *c, void *spec, bool inverse, int j0, int nj, bool f64) {
  const int T = c->pp.ztile;
#define PTC_CASE(N, TT) \
  if (c->nz == N && T == TT) return z_t<N, TT>(c, spec, inverse, j0, nj, f64);
  PTC_Z_SIZES(PTC_CASE)
  PTC_Z_WIDE(PTC_CASE)
#undef PTC_CASE
  set_error("no specialised z kernel for this length and tile");
  return PTC_E_UNSUPPORTED;
}

}  // namespace ptc
