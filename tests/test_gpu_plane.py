"""Fused passes over 2-D fields against the oracle, bit for bit: every pass
depth, every sign branch, rows narrower than a lane pair, a tile and the
halo, odd and even widths (one access per lane or two), few and many rows,
fields at addresses that only one value is aligned to, fields past the
Infinity Cache (streaming stores), NaN and Inf."""
from __future__ import annotations

import ctypes as C
import itertools

import numpy as np
import pytest

from conftest import bits

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

SHAPES = [(40, 130), (37, 121), (9, 3), (1, 250), (5, 1), (2, 2), (300, 64), (23, 247)]
SIGNS = list(itertools.product((1, -1), repeat=2))


@pytest.mark.parametrize("dtype", ["f64", "f32", "bf16"])
@pytest.mark.parametrize("shape", SHAPES)
def test_plane_passes_bit_exact(oracle, dtype, shape):
    from fidibench_amd import Upwind, configs as K
    f0 = oracle.uniform(shape, -0.5, 1.0, seed=sum(shape))
    for signs in SIGNS:
        v = (0.4 * signs[0], 0.3 * signs[1])
        dt = K.cfl_dt(shape, v, (1.0, 1.0))
        with Upwind(v, (1, 1), shape, dtype=dtype) as up:
            up.set_field(f0)
            start = up.get_field()
            ref = oracle.advect(start, v, (1, 1), dt, 19)
            for k in (0, 2, 3, 4, 5, 6, 7, 8):
                up.set_time_block(k)
                up.set_field(f0)
                plan = up.plan_passes(19, dt, k)
                ms, launches = up.advect_timed(19, dt)
                assert launches == len(plan) and sum(plan) == 19
                assert np.array_equal(bits(up.get_field()), bits(ref)), (shape, signs, k)


@pytest.mark.parametrize("dtype,offset", [("f64", 1), ("f32", 1), ("f32", 2), ("bf16", 1)])
def test_plane_pass_on_barely_aligned_fields(dtype, offset):
    from fidibench_amd import _lib as L
    shape, v, dt = (50, 140), (-0.4, 0.3), 1e-3
    n = shape[0] * shape[1]
    tdt = {"f64": torch.float64, "f32": torch.float32, "bf16": torch.bfloat16}[dtype]
    f0 = torch.rand(n, device="cuda").to(tdt)

    def run(off, k):
        a, b = (torch.zeros(n + 8, dtype=tdt, device="cuda")[off:off + n] for _ in range(2))
        a.copy_(f0)
        r = C.c_int()
        L.check(L.lib().fdb_advect_dev(2, L.u64s(shape), L.dbls(v), L.dbls((1, 1)), dt,
                                       L.DTYPES[dtype], a.data_ptr(), b.data_ptr(), 8, k,
                                       torch.cuda.current_stream().cuda_stream, C.byref(r)))
        return (b if r.value else a).clone()

    assert torch.equal(run(offset, 8), run(0, 1))


def test_plane_pass_beyond_the_cache():
    from fidibench_amd import Upwind
    shape, v, dt = (4200, 4101), (0.4, -0.3), 1e-4
    out = []
    for k in (1, 5):
        with Upwind(v, (1, 1), shape) as up:
            up.init_field(1, (0.5, 0.5, 0.5, 0.25, 0.01), seed=4)
            up.set_time_block(k)
            up.advect(5, dt)
            out.append(up.get_field())
    assert np.array_equal(bits(out[0]), bits(out[1]))


def test_plane_pass_keeps_nan_and_inf_where_the_steps_put_them(oracle):
    from fidibench_amd import Upwind
    shape, v, dt = (33, 150), (0.4, 0.3), 1e-3
    f0 = oracle.uniform(shape, 0.0, 1.0, seed=1)
    f0[3, 149], f0[30, 7], f0[0, 0] = np.nan, np.inf, -np.inf
    got = []
    for k in (1, 8):
        with Upwind(v, (1, 1), shape) as up:
            up.set_field(f0)
            up.set_time_block(k)
            up.advect(8, dt)
            got.append(up.get_field())
    assert np.array_equal(np.isnan(got[0]), np.isnan(got[1]))
    ok = ~np.isnan(got[0])
    assert np.array_equal(got[0][ok], got[1][ok])
