"""The velocity and pressure update by pairs of points at the edges of its
blocks: rows of 4 to 160 pairs (blocks 32 and 64 pairs wide), row counts that
leave part of a block idle, the smallest plane count, blocks of 128 threads
against the oracle, to the bar of the kernel tests."""
import numpy as np
import pytest

from oracle.oracle import Oracle
from paratc_amd import capi as F
from paratc_amd.solver import Solver
from helpers import inner, rel_err
from test_gpu_tscheme import TOL, rand_state, small_channel, upload_state

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("grid", [(8, 4, 8), (10, 6, 14), (64, 10, 8), (70, 14, 18), (126, 8, 10), (140, 6, 36),
                                  (256, 30, 20), (320, 50, 28)], ids=lambda g: "x".join(map(str, g)))
def test_update_matches_oracle(grid):
    case = small_channel(*grid)
    orc = Oracle(case)
    ux, uy, uz, p, _ = rand_state(case, orc, seed=3)
    orc.PMcoeUpdate(3, 2e-3)
    phi = np.asfortranarray(np.random.default_rng(4).standard_normal(ux.shape))
    orc.SetBC_and_UpdateHalo_pr(phi)
    refs = [a.copy(order="F") for a in (ux, uy, uz, p)]
    orc.FluidVelUpdate(phi, *refs[:3])
    orc.PressureUpdate(refs[3], phi)
    with Solver(case) as s:
        upload_state(s, ux, uy, uz, p)
        s.upload(F.F_HALO, phi)
        s.PMcoeUpdate(3, 2e-3)
        s.FluidVelUpdate(F.F_HALO, F.F_UX, F.F_UY, F.F_UZ)
        s.PressureUpdate(F.F_PR, F.F_HALO)
        for fid, ref in zip((F.F_UX, F.F_UY, F.F_UZ, F.F_PR), refs):
            assert rel_err(s.download(fid, F.L_INTERIOR), inner(ref)) <= TOL
