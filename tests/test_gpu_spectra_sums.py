"""The spectra's partial sums at the lengths where their launch changes: one to
four kx per thread, several segments of kx, part-filled kz chunks, the row ny+1 of
uy in the cell-centre spectrum (random ghost rows).  1e-12 of each quantity's
largest value, as for the other lengths.
"""
import pytest

from paratc_amd import case as CS
from test_gpu_spectra import TOL, run_case
from test_gpu_tscheme import small_channel

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("grid", [(16, 4, 18), (126, 6, 10), (640, 4, 12), (1400, 4, 8), (2500, 4, 8), (2700, 6, 8)],
                         ids=lambda g: "x".join(map(str, g)))
@pytest.mark.parametrize("half", [False, True])
def test_sums_match_oracle(grid, half):
    case = small_channel(*grid)
    case.is_use_crf, case.ucrf_in = True, 0.3
    if half:
        case.flow_type = CS.FT_HC
    r = run_case(case, 41, jlcs=2, rows=(2, grid[1] // 2), samples=2)
    assert r["ex"] <= TOL and r["ez"] <= TOL and r["e2"] <= TOL, r
    assert r["n"] == 2 and r["reset"]
