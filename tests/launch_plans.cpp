// Host-side launch plans of the library printed for tests/test_launch_plans.py
// (no device is touched): one plan per line, the first word its kind.
#include <cstdio>

#include "ptc_internal.hpp"

namespace ptc {
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
  return 0;
}
