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
  return 0;
}
