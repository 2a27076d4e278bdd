"""The refinement's residual by columns of planes: every length that has the
form, groups of 8 and of 4 planes, rows next to a wall, tiles of one row, plane
counts whose tiles hold no whole group (the pair-by-pair form), slabs.

A wrong residual does not converge to the FP64 solution.  Bars as for the other
FP32-storage grids: each sweep gains two orders until the accuracy of an FP64
residual, 1e-11 relative, 5e-10 for rows of 1024 points and more.
"""
import pytest

from oracle.oracle import Oracle
from paratc_amd import capi, case as CS, ic
from paratc_amd.solver import Solver

from helpers import inner, rel_err

pytestmark = pytest.mark.gpu

GRIDS = [
    (16, 16, 16, 0),    # 8 pairs a row, 32 lines a workgroup
    (32, 16, 32, 0),
    (64, 20, 16, 0),
    (128, 18, 64, 9),   # slabs whose tiles are one row
    (256, 24, 16, 0),
    (256, 24, 16, 8),   # slabs
    (512, 16, 16, 0),
    (1024, 16, 32, 0),  # groups of four planes
    (64, 16, 700, 0),   # tiles of four planes: pair by pair
    (96, 16, 32, 0),    # a length without the form
]

@pytest.mark.parametrize("grid", GRIDS, ids=lambda g: "x".join(map(str, g)))
def test_refinement_converges(grid):
    nx, ny, nz, slab = grid
    case = CS.case_poisson(nx, ny, nz, 1.8)
    f = ic.poisson_rhs(case, seed=7)
    orc = Oracle(case)
    ref = orc.halo()
    orc.clcPPE(f.copy(order="F"), ref, 1)
    errs = []
    with Solver(case) as s:
        s.upload(capi.F_ARR1, f, capi.L_INTERIOR)
        for sweeps in (0, 1, 3):
            s.poisson_config(capi.PREC_FP32_REFINE, capi.TRI_AUTO, 0, sweeps)
            if slab:
                s.poisson_slab_planes(slab)
            s.clcPPE(capi.F_ARR1, capi.F_HALO)
            errs.append(rel_err(s.download(capi.F_HALO, capi.L_INTERIOR), inner(ref)))
    print(grid, [f"{e:.1e}" for e in errs], flush=True)
    assert errs[0] < 1e-4
    assert errs[1] < 1e-2 * errs[0]
    assert errs[2] <= (1e-11 if nx < 1024 else 5e-10)
