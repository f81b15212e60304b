"""2-D fields beyond the caches (streaming stores), at addresses that only one
value is aligned to, and with NaN and Inf, each against the oracle's steps:
one-step launches are the plane kernel's too, so comparing pass depths with
each other is no check of what they share."""
from __future__ import annotations

import ctypes as C

import numpy as np
import pytest

from conftest import bits

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.mark.parametrize("v", [(0.4, -0.3), (-0.2, 0.3)])
@pytest.mark.parametrize("width", [4101, 4102])
def test_steps_beyond_the_cache_equal_the_oracle(oracle, v, width):
    from fidibench_amd import Upwind
    shape, dt = (4200, width), 1e-4
    f0 = oracle.uniform(shape, -0.5, 1.0, seed=width)
    ref = oracle.advect(f0, v, (1, 1), dt, 3)
    with Upwind(v, (1, 1), shape) as up:
        for k in (1, 2, 3):
            up.set_field(f0)
            up.set_time_block(k)
            up.advect(3, dt)
            assert np.array_equal(bits(up.get_field()), bits(ref)), k


@pytest.mark.parametrize("dtype", ["f64", "f32", "bf16"])
@pytest.mark.parametrize("width", [150, 151])
def test_nan_and_inf_equal_the_oracle(oracle, dtype, width):
    from fidibench_amd import Upwind
    shape, v, dt = (33, width), (0.4, -0.3), 1e-3
    f0 = oracle.uniform(shape, 0.0, 1.0, seed=1)
    f0[3, width - 1], f0[30, 7], f0[0, 0] = np.nan, np.inf, -np.inf
    with Upwind(v, (1, 1), shape, dtype=dtype) as up:
        up.set_field(f0)
        with np.errstate(all="ignore"):
            ref = oracle.advect(up.get_field(), v, (1, 1), dt, 8)
        wide = _wide(ref)
        for k in (1, 2, 5, 8):
            up.set_field(f0)
            up.set_time_block(k)
            up.advect(8, dt)
            got = up.get_field()
            assert np.array_equal(np.isnan(_wide(got)), np.isnan(wide)), k
            ok = ~np.isnan(wide)
            assert np.array_equal(bits(got)[ok], bits(ref)[ok]), k


def _wide(a):
    if a.dtype == np.uint16:
        return (a.astype(np.uint32) << 16).view(np.float32)
    return a


@pytest.mark.parametrize("dtype,offset", [("f64", 1), ("f32", 1), ("f32", 2)])
@pytest.mark.parametrize("k", [1, 4])
def test_barely_aligned_fields_equal_the_oracle(oracle, dtype, offset, k):
    from fidibench_amd import _lib as L
    shape, v, dt = (50, 140), (-0.4, 0.3), 1e-3
    n = shape[0] * shape[1]
    ndt, tdt = {"f64": (np.float64, torch.float64), "f32": (np.float32, torch.float32)}[dtype]
    f0 = oracle.uniform(shape, 0.0, 1.0, seed=2).astype(ndt)
    a, b = (torch.zeros(n + 8, dtype=tdt, device="cuda")[offset:offset + n] for _ in range(2))
    a.copy_(torch.from_numpy(f0.reshape(-1)))
    r = C.c_int()
    L.check(L.lib().fdb_advect_dev(2, L.u64s(shape), L.dbls(v), L.dbls((1, 1)), dt,
                                   L.DTYPES[dtype], a.data_ptr(), b.data_ptr(), 4, k,
                                   torch.cuda.current_stream().cuda_stream, C.byref(r)))
    got = (b if r.value else a).cpu().numpy().reshape(shape)
    assert np.array_equal(bits(got), bits(oracle.advect(f0, v, (1, 1), dt, 4)))
