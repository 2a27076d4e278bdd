"""The Poisson source formed by columns of planes in the specialised x pass:
plane counts that are and are not multiples of the groups of 4 and 2 planes,
row counts of every tile, lengths whose lines do not fill a workgroup.
One step against the oracle: 1e-12 per velocity field, divergence 1e-10 and its
maximum before the solve, the bars of the step tests."""
import pytest

from paratc_amd import capi
from helpers import rel_err
from test_gpu_tscheme import inner_y, run_iterate, small_channel

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("grid", [(16, 6, 8), (32, 10, 18), (64, 8, 10), (96, 6, 30), (128, 12, 14), (192, 4, 14),
                                  (256, 4, 18), (512, 4, 10), (1024, 4, 14), (1536, 4, 10)],
                         ids=lambda g: "x".join(map(str, g)))
def test_step_with_the_source_by_columns(grid):
    nx, ny, nz = grid
    case = small_channel(nx, ny, nz)
    plan = lambda s: s.poisson_config(capi.PREC_FP64, capi.TRI_AUTO, 0, 0)
    out, ref, mons, _, _ = run_iterate(case, 1, plan=plan)
    for f in (0, 1, 2):
        assert rel_err(inner_y(out[f]), inner_y(ref[f])) <= 1e-12
    mo, mg = mons[-1]
    assert mg[1] <= 1e-10 and abs(mg[0] - mo[0]) <= 1e-11
