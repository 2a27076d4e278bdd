"""clcStat's row-marching sums against the oracle at the shapes where the launch
changes: rows shorter than a wavefront, several rows per workgroup with the last
group part-filled, rows of exactly one workgroup, rows in two and three segments
with part-filled ends, z chunks with a remainder.

Each statistic is a mean of at most a few 1e5 products of O(1) values in both
orders of summation, so 1e-12 of its largest value over j holds by a wide margin.
"""
import numpy as np
import pytest

from helpers import random_halo
from oracle.oracle import Oracle
from paratc_amd import capi, case as CS
from paratc_amd import ensemble as E
from paratc_amd.solver import Solver

pytestmark = pytest.mark.gpu

GRIDS = [(8, 4, 8), (36, 6, 18), (64, 10, 50), (96, 14, 36), (128, 6, 28), (256, 4, 16), (270, 6, 10), (504, 4, 8),
         (512, 6, 14), (1024, 4, 18)]


@pytest.mark.parametrize("grid", GRIDS, ids=lambda g: "x".join(map(str, g)))
@pytest.mark.parametrize("kind", ["channel", "scalar", "half"])
def test_stat_rows_match_oracle(grid, kind):
    nx, ny, nz = grid
    case = (E.case_channel_scalar(nx, ny, nz, re_b=3000.0, ws=0.02) if kind == "scalar"
            else CS.case_channel(nx, ny, nz, 1.7))
    if kind == "half":
        case.flow_type, case.yly = CS.FT_HC, 1.0
        case.ny = ny + 1
        case.sections = [CS.MeshSection(1.0, ny + 1, 1, 0, 1.7)]
        case.is_use_crf, case.ucrf_in = True, 0.2
    orc = Oracle(case)
    ns = 40 if case.scalar else 35
    ref = np.zeros((ns, case.ny + 1), order="F")
    f = [random_halo((nx, case.ny, nz), 50 + q) for q in range(5)]
    orc.clcStat(*f, ref)
    with Solver(case) as s:
        for fid, a in zip((capi.F_UX, capi.F_UY, capi.F_UZ, capi.F_PR, capi.F_SCALAR), f):
            if fid != capi.F_SCALAR or case.scalar:
                s.upload(fid, a)
        s.clcStat()
        one, _, _ = s.get_stat()
        s.clcStat()
        two, nf, _ = s.get_stat()
    scale = np.maximum(np.abs(ref).max(axis=1, keepdims=True), 1e-300)
    assert nf == 2
    assert (np.abs(one - ref) / scale).max() <= 1e-12
    assert (np.abs(two - 2 * ref) / scale).max() <= 2e-12


@pytest.mark.parametrize("ny", [7, 31])  # 320 values and one more; 1280, a whole number of workgroups
def test_stat_read_and_reset(ny):
    case = E.case_channel_scalar(16, ny + 1, 8, re_b=3000.0, ws=0.02)
    case.flow_type, case.yly, case.ny = CS.FT_HC, 1.0, ny
    case.sections = [CS.MeshSection(1.0, ny, 1, 0, 1.7)]
    with Solver(case) as s:
        none, nf, pg = s.get_stat(reset=True)
        assert not none.any() and nf == 0 and pg == 0.0
        for q, fid in enumerate((capi.F_UX, capi.F_UY, capi.F_UZ, capi.F_PR, capi.F_SCALAR)):
            s.upload(fid, random_halo((16, ny, 8), 70 + q))
        s.clcStat()
        one, nf, _ = s.get_stat()
        kept, nf1, _ = s.get_stat(reset=True)
        assert nf == nf1 == 1 and one[:, :ny].all() and np.array_equal(one, kept)
        gone, nf2, pg2 = s.get_stat()
        assert not gone.any() and nf2 == 0 and pg2 == 0.0
        s.clcStat()
        again, _, _ = s.get_stat()
        assert np.array_equal(again, one)
