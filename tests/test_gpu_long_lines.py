"""The run-time length x passes at the lines of one workgroup each: the longest
that are padded and unpadded (h = nx/2 = 3600, 3675, 4096), and time steps whose
source is formed by workgroups of more than 256 threads, against the oracle.

Bars: 1e-12 relative for a solve and, after a step, per velocity field, as for
the other lengths.
"""
import numpy as np
import pytest

from oracle.oracle import Oracle
from paratc_amd import capi, case as CS, ic
from paratc_amd.solver import Solver
from test_gpu_tscheme import inner_y, rel_err, run_iterate, small_channel
from helpers import inner

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("grid", [(7200, 4, 8), (7350, 4, 8), (8192, 4, 8)], ids=lambda g: "x".join(map(str, g)))
def test_longest_lines_match_oracle(grid):
    case = CS.case_poisson(*grid, 1.7)
    f = ic.poisson_rhs(case, seed=31)
    orc = Oracle(case)
    ref = orc.halo()
    orc.clcPPE(f.copy(order="F"), ref, 1)
    with Solver(case) as s:
        s.poisson_config(capi.PREC_FP64, capi.TRI_AUTO, 0, 0)
        s.upload(capi.F_ARR1, f, capi.L_INTERIOR)
        s.clcPPE(capi.F_ARR1, capi.F_HALO)
        out = s.download(capi.F_HALO, capi.L_INTERIOR)
    assert rel_err(out, inner(ref)) <= 1e-12


@pytest.mark.parametrize("grid", [(1372, 6, 12), (2304, 4, 10), (8192, 4, 8)], ids=lambda g: "x".join(map(str, g)))
def test_step_with_one_line_per_workgroup(grid):
    def plan(s):
        s.poisson_config(capi.PREC_FP64, capi.TRI_AUTO, 0, 0)

    out, ref, mons, _, _ = run_iterate(small_channel(*grid), 1, plan=plan)
    for f in (capi.F_UX, capi.F_UY, capi.F_UZ):
        assert np.isfinite(out[f]).all()
        assert rel_err(inner_y(out[f]), inner_y(ref[f])) <= 1e-12
    mo, mg = mons[-1]
    # (the divergence before the projection is of the order of the noise over dx)
    assert mg[1] <= 1e-10 and abs(mg[0] - mo[0]) <= 1e-12 * max(1.0, mo[0])
