"""Stored states of a gradient by four-step store-all passes (FP32 and FP64)
against one launch per step: the same states and lam bit for bit, for tiles
cut on each axis, both directions of each axis, runs that leave 0 to 3 single
steps, and grids of at most one tile."""
from __future__ import annotations

import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


# tiles of 60 x 44 (FP32) and 60 x 28 (FP64) cells
@pytest.mark.parametrize("shape", [(3, 5, 7), (12, 44, 60), (13, 45, 61), (9, 28, 121),
                                   (40, 29, 59), (96, 96, 96)])
@pytest.mark.parametrize("v", [(0.45, 0.3, 0.2), (-0.3, 0.45, -0.2), (0.4, -0.35, 0.25),
                               (-0.45, -0.3, -0.2)])
@pytest.mark.parametrize("dtype", ["f64", "f32"])
@pytest.mark.parametrize("T", [5, 8, 12])
def test_stored_states_equal_one_step_launches(shape, v, dtype, T):
    from fidibench_amd import _lib as L
    from fidibench_amd.autograd import Tape
    code, tdt = {"f64": (L.F64, torch.float64), "f32": (L.F32, torch.float32)}[dtype]
    g = torch.Generator(device="cuda").manual_seed(T)
    f0 = torch.rand(shape, generator=g, device="cuda", dtype=tdt)
    lamT = torch.randn(shape, generator=g, device="cuda", dtype=tdt)
    out = []
    for k in (8, 4, 1):
        tape = Tape(shape, v, (1, 1, 1), 2e-3, T, code, code, 1 << 30)
        tape.set_time_block(k)
        fT, lam0 = torch.empty_like(f0), torch.empty_like(f0)
        tape.forward(f0, fT)
        gv = tape.backward(lamT, lam0)
        assert tape.stats()["forward_steps"] == T
        tape.close()
        out.append((fT, lam0, gv))
    for fT, lam0, gv in out[:2]:
        assert torch.equal(fT, out[2][0]) and torch.equal(lam0, out[2][1])
        # The products see every stored state: sums of the same cells' terms
        # in another order, each within 2^-50 of its size (compensated).
        scale = max(abs(x) for x in out[2][2])
        assert all(abs(a - b) <= 1e-12 * scale for a, b in zip(gv, out[2][2]))
