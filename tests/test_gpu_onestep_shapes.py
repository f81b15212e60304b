"""One-step launches on both sides of the rules that pick their shape: a
grid with fewer tiles than the launch wants blocks (one plane per block),
fields that fit the Infinity Cache with and without the streaming stores
(40 MiB and 256 MiB of fields read and written), ragged axes.  Forward and
transpose against the oracle bit for bit; the velocity products to 1e-11 of
the sum of their magnitudes (compensated FP64 sums of the same products)."""
from __future__ import annotations

import numpy as np
import pytest

from conftest import bits

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

# FP64 in + out: 0.5 MB (32 planes, 2 tiles), 39 MiB, 42 MiB, 255 MiB, 258 MiB.
SHAPES = [(32, 24, 40), (101, 113, 224), (109, 121, 209), (235, 263, 270), (241, 260, 270)]


@pytest.mark.parametrize("shape", SHAPES)
@pytest.mark.parametrize("dtype", ["f64", "f32", "bf16", "bf16sr"])
def test_one_step_bit_exact_across_shape_rules(oracle, shape, dtype):
    from fidibench_amd import Upwind, configs as K
    v = (0.3, -0.45, 0.2)
    dt = K.cfl_dt(shape, v)
    f0 = oracle.uniform(shape, 0.0, 1.0, seed=sum(shape))
    with Upwind(v, (1, 1, 1), shape, dtype=dtype) as up:
        up.set_field(f0)
        start = up.get_field()
        if dtype == "bf16sr":
            up.set_seed(5)
            ref = oracle.advect_bf16_sr(start, v, (1, 1, 1), dt, 2, seed=5)
        else:
            ref = oracle.advect(start, v, (1, 1, 1), dt, 2)
        up.advect(2, dt)
        assert np.array_equal(bits(up.get_field()), bits(ref))


@pytest.mark.parametrize("shape", SHAPES[:3] + [(190, 240, 245)])
def test_adjoint_step_bit_exact_across_shape_rules(oracle, shape):
    from fidibench_amd import _lib as L
    v, one, dt = (-0.3, 0.45, 0.2), (1.0, 1.0, 1.0), 0.01
    lam_next = oracle.uniform(shape, -1, 1, seed=3)
    f = oracle.uniform(shape, 0, 1, seed=4)
    ref = oracle.adjoint(lam_next, v, one, dt, 1)
    terms = oracle.vgrad_terms(lam_next, f, v, one, dt)
    a, ft = torch.from_numpy(lam_next).cuda(), torch.from_numpy(f).cuda()
    b, acc = torch.empty_like(a), torch.zeros(6, dtype=torch.float64, device="cuda")
    L.check(L.lib().fdb_adjoint_step_dev(3, L.u64s(shape), L.dbls(v), L.dbls(one), dt, L.F64,
                                         a.data_ptr(), b.data_ptr(), L.F64, ft.data_ptr(),
                                         acc.data_ptr(), torch.cuda.current_stream().cuda_stream))
    torch.cuda.synchronize()
    assert np.array_equal(bits(b.cpu().numpy()), bits(ref))
    s = acc.cpu().numpy()
    for j in range(3):
        up = 1 if v[j] < 0 else -1
        scale = float(np.abs(lam_next * (np.roll(f, -up, j) - f)).sum())
        assert abs(s[2 * j] + s[2 * j + 1] - terms[j]) <= 1e-11 * scale


# Up to four rows a plane: blocks of two waves of two rows.
FEW_ROWS = [(1,), (63,), (131303,), (5, 1, 130), (3, 2, 65), (40, 3, 257), (9, 4, 1000), (9, 5, 96)]


@pytest.mark.parametrize("shape", FEW_ROWS)
@pytest.mark.parametrize("dtype", ["f64", "f32", "bf16", "bf16sr"])
def test_one_step_bit_exact_with_few_rows(oracle, shape, dtype):
    from fidibench_amd import Upwind, configs as K
    for sign in (1.0, -1.0):
        v, one = tuple(sign * x for x in (0.3, -0.45, 0.2)[:len(shape)]), (1.0,) * len(shape)
        dt = K.cfl_dt(shape, v)
        f0 = oracle.uniform(shape, 0.0, 1.0, seed=sum(shape))
        with Upwind(v, one, shape, dtype=dtype) as up:
            up.set_field(f0)
            start = up.get_field()
            if dtype == "bf16sr":
                up.set_seed(5)
                ref = oracle.advect_bf16_sr(start, v, one, dt, 2, seed=5)
            else:
                ref = oracle.advect(start, v, one, dt, 2)
            up.advect(2, dt)
            assert np.array_equal(bits(up.get_field()), bits(ref))


@pytest.mark.parametrize("shape", [(9, 1, 130), (30, 2, 65), (7, 4, 301), (1, 3, 5000)])
def test_adjoint_step_bit_exact_with_few_rows(oracle, shape):
    test_adjoint_step_bit_exact_across_shape_rules(oracle, shape)
