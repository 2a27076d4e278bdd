"""The run-time length FFT passes against the oracle: plans of one to four
stages, every radix from 2 to 10 and the radix-15 fallback, lines that do not
fill a workgroup, workgroups of one long line, narrow z tiles.

The bar is the Poisson solve's 1e-12 relative, and after one time step 1e-12
per velocity field, as for the specialised lengths.
"""
import numpy as np
import pytest

from oracle.oracle import Oracle
from paratc_amd import capi, case as CS, ic
from paratc_amd.solver import Solver
from test_gpu_tscheme import inner_y, rel_err, run_iterate, small_channel
from helpers import inner

pytestmark = pytest.mark.gpu

# (nx, ny, nz) and the stages of nx/2; nz
GRIDS = [
    (8, 4, 8),      # 4; 8
    (18, 6, 10),    # 9; 10
    (14, 6, 84),    # 7; 84 = 7 * 4 * 3
    (98, 8, 126),   # 7 * 7; 7 * 6 * 3
    (250, 6, 250),  # 5 * 5 * 5; 10 * 5 * 5
    (360, 10, 150),  # 6 * 6 * 5; 6 * 5 * 5
    (162, 12, 42),  # 9 * 9; 7 * 6
    (2000, 4, 18),  # 10 * 10 * 10; 9 * 2
    (5400, 4, 10),  # h = 2700: one line of several hundred threads per workgroup
    (6750, 4, 8),   # h = 3375 = 15 * 15 * 15
    (16, 4, 3750),  # one-column tiles of 750 threads
    (22, 4, 1200),  # nx / 2 = 11 is refused
]


@pytest.mark.parametrize("grid", GRIDS[:-1], ids=lambda g: "x".join(map(str, g)))
@pytest.mark.parametrize("tile", [0, 2])
def test_lengths_match_oracle(grid, tile):
    nx, ny, nz = grid
    case = CS.case_poisson(nx, ny, nz, 1.7)
    f = ic.poisson_rhs(case, seed=12)
    orc = Oracle(case)
    ref = orc.halo()
    orc.clcPPE(f.copy(order="F"), ref, 1)
    with Solver(case) as s:
        s.poisson_config(capi.PREC_FP64, capi.TRI_AUTO, tile, 0)
        s.upload(capi.F_ARR1, f, capi.L_INTERIOR)
        s.clcPPE(capi.F_ARR1, capi.F_HALO)
        out = s.download(capi.F_HALO, capi.L_INTERIOR)
        assert np.array_equal(s.download(capi.F_ARR1, capi.L_INTERIOR), f)
    assert rel_err(out, inner(ref)) <= 1e-12


def test_other_factors_stay_refused():
    with pytest.raises((capi.PtcError, ValueError)):
        Solver(CS.case_poisson(*GRIDS[-1], 1.7))


@pytest.mark.parametrize("grid", [(36, 20, 30), (50, 12, 14), (180, 6, 42)], ids=lambda g: "x".join(map(str, g)))
def test_step_forms_its_source_in_the_x_pass(grid):
    """A time step on lengths without a compiled kernel: the divergence formed
    in the run-time x pass, its maximum, and the ghost rows of the inverse."""
    out, ref, mons, _, _ = run_iterate(small_channel(*grid), 1)
    for fid in (capi.F_UX, capi.F_UY, capi.F_UZ):
        assert rel_err(inner_y(out[fid]), inner_y(ref[fid])) <= 1e-12
    mo, mg = mons[-1]
    assert mg[1] <= 1e-10 and abs(mg[0] - mo[0]) <= 1e-11
