"""The partitioned y-solves at the edges of the reduced system: one, two and
three chunks, chunk counts next to a power of two, padded last chunks, every
kernel form, against the oracle (1e-12 relative, the
bar of a solve and of the velocities after a step)."""
import numpy as np
import pytest

from oracle.oracle import Oracle
from paratc_amd import capi, case as CS, ic
from paratc_amd.solver import Solver
from helpers import inner, rel_err

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("form", ["complex16", "complex32", "lds16", "lanes64", "lanes32"])
@pytest.mark.parametrize("ny,rows", [(4, 4), (8, 8), (10, 8), (12, 4), (16, 8), (24, 8), (30, 4), (34, 8), (36, 4),
                                     (36, 12), (48, 16)])
def test_poisson_chunks(ny, rows, form):
    case = CS.case_poisson(16, ny, 12, 1.7)
    f = ic.poisson_rhs(case, seed=3)
    orc = Oracle(case)
    ref = orc.halo()
    orc.clcPPE(f.copy(order="F"), ref, 1)
    with Solver(case) as s:
        s.poisson_config(capi.PREC_FP64, capi.TRI_AUTO, 0, 0)
        s.upload(capi.F_ARR1, f, capi.L_INTERIOR)
        n = int("".join(ch for ch in form if ch.isdigit()))
        try:
            s.poisson_chunk_rows(rows)
            {"complex": s.poisson_tri_complex, "lds": s.poisson_tri_lines,
             "lanes": s.poisson_tri_lanes}[form.rstrip("0123456789")](n)
        except capi.PtcError as e:
            assert "tridiagonal kernel" in str(e)  # no such shape for this ny
            pytest.skip("no such shape")
        if s.poisson_get_config()["tri"] != "partitioned":
            pytest.skip("no such shape")
        assert s.poisson_get_config()["chunk_rows"] == rows
        s.clcPPE(capi.F_ARR1, capi.F_HALO)
        out = s.download(capi.F_HALO, capi.L_INTERIOR)
    assert rel_err(out, inner(ref)) <= 1e-12


@pytest.mark.parametrize("ny", [4, 12, 14, 24, 26, 38, 100])
def test_crank_nicolson_chunks(ny):
    """u, v, w after an AB2 step."""
    from test_gpu_tscheme import inner_y, run_iterate
    case = CS.case_channel(16, ny, 12, 1.7)
    case.ischeme = 1
    out, ref, _, _, _ = run_iterate(case, 1)
    for f in (0, 1, 2):
        assert np.isfinite(out[f]).all()
        assert rel_err(inner_y(out[f]), inner_y(ref[f])) <= 1e-12
