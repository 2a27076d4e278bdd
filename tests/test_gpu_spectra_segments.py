"""The spectra's partial sums where the kx of a row just pass a workgroup's share:
two kx per thread from 257 on (512 points), a second segment of one kx at 1025
(2048 points).  1e-12 of each quantity's largest value, as for the other lengths.
"""
import pytest

from test_gpu_spectra import TOL, run_case
from test_gpu_tscheme import small_channel

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("grid", [(500, 4, 18), (512, 4, 18), (2000, 4, 8), (2048, 4, 8)],
                         ids=lambda g: "x".join(map(str, g)))
def test_sums_match_oracle(grid):
    case = small_channel(*grid)
    case.is_use_crf, case.ucrf_in = True, 0.3
    r = run_case(case, 43, jlcs=2, rows=(2, grid[1] // 2), samples=2)
    assert r["ex"] <= TOL and r["ez"] <= TOL and r["e2"] <= TOL, r
    assert r["n"] == 2 and r["reset"]
