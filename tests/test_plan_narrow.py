"""The planner over grids whose rows are short: a one-step launch costs by the
rows it issues there, not by its bytes, and several steps a launch are cheaper
(launch times measured on MI355X)."""
from __future__ import annotations

import pytest


def _passes(dtype, shape, nsteps=22):
    from fidibench_amd import _lib as L
    v = (0.4, -0.3, 0.35)[:len(shape)]
    return L.plan_passes(shape, v, (1.0,) * len(shape), 1e-6, getattr(L, dtype), nsteps, 0)


@pytest.mark.parametrize("dtype,shape", [
    ("F64", (1256, 3519, 2)),   # us a step, one a launch / fused: 537 / 127
    ("F32", (1256, 3519, 2)),   # 313 / 68
    ("BF16", (1256, 3519, 2)),  # 339 / 86
    ("F64", (200, 300, 1)),     # 10.9 / 2.6
    ("F32", (74, 6433, 9)),     # 56 / 13
    ("BF16", (400, 400, 16)),   # 16.7 / 4.1
    ("BF16", (300507, 14)),     # 62 / 9
    ("F32", (2077634, 3)),      # 243 / 44
    ("BF16", (3000, 3000, 16)),  # 790 / 172, above 512^3 cells
    ("F64", (5000, 9000, 4)),   # 5259 / 1229
])
def test_short_rows_take_several_steps_a_launch(dtype, shape):
    assert 1 not in _passes(dtype, shape)


@pytest.mark.parametrize("dtype", ["F64", "F32", "BF16"])
def test_one_step_in_one_launch(dtype):
    assert _passes(dtype, (1256, 3519, 2), 1) == [1]


@pytest.mark.parametrize("shape,deep", [
    ((104, 48, 225), True),     # us a step, one a launch / 4-step passes: 6.3 / 4.4
    ((1, 554, 2013), True),     # 7.2 / 4.8
    ((290, 38, 222), True),     # 8.4 / 5.7
    ((192, 3014, 2), True),     # 51 / 24
    ((1462, 4, 2), False),      # 5.2 / 9.8
    ((1643, 2, 2), False),      # 6.1 / 10.4
])
def test_stochastic_rounding_follows_the_grid_not_its_cells(shape, deep):
    ks = _passes("BF16_SR", shape)
    assert (1 not in ks) if deep else set(ks) == {1}, ks
