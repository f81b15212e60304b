"""The planner's split above 512^3 with the device's own occupancies: a run
stochastically rounded goes in 4-step passes (2-step ones are bound by HBM),
as measured at each of these grids; nothing is launched."""
from __future__ import annotations

import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [(512, 512, 512), (600, 620, 640), (768, 700, 640),
                               (1024, 1024, 768), (1024, 1024, 1024)])
@pytest.mark.parametrize("nsteps", [8, 20, 200])
def test_stochastic_rounding_runs_in_four_step_passes(n, nsteps):
    from fidibench_amd import _lib as L
    ks = L.plan_passes(n, (0.7, -0.4, 0.2), (1, 1, 1), 1e-4, L.DTYPES["bf16sr"], nsteps, 0)
    assert sum(ks) == nsteps and set(ks) == {4}
