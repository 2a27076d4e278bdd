"""The constant-flow-rate correction formed inside the Crank-Nicolson launch, on
tall channels: 13, 14, 15 and 16 chunks of 16 rows x 32 lanes (416 to 512
threads, the odd counts ending in half a wavefront), against the oracle.

Bars: those of a step at other heights, 1e-12 relative per velocity field and
for the pressure gradient of the substeps.
"""
import numpy as np
import pytest

from paratc_amd import capi
from test_gpu_tscheme import inner_y, rel_err, run_iterate, small_channel, small_gravity

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind", ["channel", "gravity"])
@pytest.mark.parametrize("ny", [194, 200, 208, 210, 226, 230, 240, 256])
def test_constant_flow_rate_on_tall_channels(ny, kind):
    case = small_channel(16, ny, 8) if kind == "channel" else small_gravity(16, ny, 8)
    assert case.is_ux_const
    out, ref, _, coe, ocoe = run_iterate(case, 1)
    for f in (capi.F_UX, capi.F_UY, capi.F_UZ):
        assert np.isfinite(out[f]).all()
        e = rel_err(inner_y(out[f]), inner_y(ref[f]))
        print(f"{kind} ny={ny} field {f}: {e:.3e}", flush=True)
        assert e <= 1e-12
    print(f"{kind} ny={ny} PrGradAver {coe[8]:.17g} oracle {ocoe[8]:.17g}", flush=True)
    assert abs(coe[8] - ocoe[8]) <= 1e-12 * max(1.0, abs(ocoe[8]))
