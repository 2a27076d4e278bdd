// Host-side launch plans of the library printed for tests/test_launch_plans.py
// (no device is touched): one plan per line, the first word its kind.
#include <cstdio>

#include "ptc_internal.hpp"

namespace ptc {
bool fft_x_shape(const FftLen &L, size_t pad_cap, size_t lds_limit, int *lines, int *threads, int *pad, size_t *lds);
int tri_plan(int ny, size_t lds_limit, bool poisson, int mm_req, int lpb_req, int *P_out, int *mm_out, int *lpb_out);
}

int main() {
  const size_t lds = 163840;  // a gfx950 CU
  // cn: ny, chunks, chunk rows, lanes, exchanged lanes
  for (int ny = 4; ny <= 256; ++ny) {
    int P = 0, mm = 0, lpb = 0;
    if (ptc::tri_plan(ny, lds, false, 0, 0, &P, &mm, &lpb) == PTC_OK)
      std::printf("cn %d %d %d %d %d\n", ny, P, mm, lpb, ptc::cn_exchange_lanes(lpb));
  }
  // x: h, LDS limit, accepted, threads per line, lines, threads, padding shift, bytes (the
  // run-time length x passes' lines of h = nx/2 complex values)
  for (size_t limit : {size_t(65536), lds})
    for (int h = 4; h <= 4096; ++h) {
      ptc::FftLen L{};
      if (ptc::fft_make_len(h, &L) != PTC_OK) continue;
      int lines = 0, threads = 0, pad = 0;
      size_t bytes = 0;
      const bool ok = ptc::fft_x_shape(L, 65536, limit, &lines, &threads, &pad, &bytes);
      std::printf("x %d %zu %d %d %d %d %d %zu\n", h, limit, ok, L.threads, lines, threads, pad, bytes);
    }
  // rhs: nx, ny, requested segment threads and rows, LDS limit, threads per row, rows, bytes
  for (size_t limit : {size_t(65536), lds})
    for (int nx = 8; nx <= 1100; nx += 2)
      for (int ny : {4, 10, 96, 256})
        for (int seg : {0, 64, 128, 256})
          for (int rows : {0, 1, 2, 4, 8}) {
            ptc_ctx c;
            c.nx = nx;
            c.ny = ny;
            c.nz = 64;
            c.n3 = (size_t)nx * (ny + 2) * c.nz;
            c.lds_limit = limit;
            c.rhs_seg_req = seg;
            c.rhs_rows_req = rows;
            int tx = 0, ty = 0, run = 0, minpl = 0;
            ptc::rhs_shape_in_use(&c, &tx, &ty, &run, &minpl);
            std::printf("rhs %d %d %d %d %zu %d %d %zu\n", nx, ny, seg, rows, limit, tx, ty, ptc::rhs_lds_in_use(&c));
          }
  return 0;
}
