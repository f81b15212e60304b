"""checksum() and std() of fields folded on the device against the
sequential loop, bit for bit: values that round at every addition, ties
(single-precision values in a double sum), both signs with the sum passing
through zero and through binades, zeros, values far apart in magnitude,
values that are not finite, and sizes around the device path's first one
and its chunks of 2048."""
from __future__ import annotations

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _fields(n):
    r = np.random.default_rng(n)
    u = r.random(n)
    sign = np.where(r.random(n) < 0.5, -1.0, 1.0)
    ball = (np.arange(n) % 977 < 300).astype(float)
    spike = np.zeros(n)
    spike[0], spike[n // 2], spike[-1] = 1.0, 1e-320, -2.5
    nan, inf = u.copy(), u.copy()
    nan[n // 3], inf[n // 2], inf[-1] = np.nan, np.inf, -np.inf
    return {
        "positive": u,
        "noisy_ball": ball + 0.01 * u,
        "ties": r.random(n, dtype=np.float32).astype(np.float64) * 0.01,
        "halves": np.where(r.random(n) < 0.5, 0.5, 1.5) * 2.0 ** -38 + np.where(
            np.arange(n) == 0, 2.0 ** 15, 0.0),
        "both_signs": u * sign,
        "negative": -u,
        "cancel": np.concatenate([u[: n // 2], -u[: n - n // 2]]),
        "scales": sign * u * 2.0 ** r.integers(-300, 300, n),
        "spike": spike,
        "zeros": np.zeros(n) * sign,
        "tiny": u * 5e-324 * 100,
        "nan": nan,
        "inf": inf,
    }


@pytest.mark.parametrize("n", [65535, 65536, 65537, 129 * 2048 - 1, 300 * 2048 + 5])
def test_folds_equal_the_sequential_loop(oracle, n):
    from fidibench_amd import Upwind
    with np.errstate(all="ignore"):
        for name, f in _fields(n).items():
            with Upwind((1.0,), (1.0,), (n,)) as up:
                up.set_field(f)
                for got, want in ((up.checksum(), oracle.checksum(f)), (up.std(), oracle.std(f))):
                    same = np.float64(got).tobytes() == np.float64(want).tobytes()
                    assert same or (np.isnan(got) and np.isnan(want)), (name, n, got, want)


@pytest.mark.parametrize("dtype", ["f32", "bf16"])
def test_folds_of_narrow_storage(oracle, dtype):
    from fidibench_amd import Upwind
    shape = (61, 70, 83)
    f = oracle.uniform(shape, -0.2, 1.0, seed=9)
    with Upwind((1.0, 1.0, 1.0), (1.0, 1.0, 1.0), shape, dtype=dtype) as up:
        up.set_field(f)
        wide = up.get_field("f64")
        assert up.checksum() == oracle.checksum(wide)
        assert up.std() == oracle.std(wide)


def test_fold_of_a_long_field(oracle):
    """Chunks longer than one tile: 2^25 + 3 values fold in chunks of 4096."""
    from fidibench_amd import Upwind
    n = 2 ** 25 + 3
    f = oracle.uniform((n,), 0.0, 1.0, seed=3)
    with Upwind((1.0,), (1.0,), (n,)) as up:
        up.set_field(f)
        assert up.checksum() == oracle.checksum(f)


def test_filter_checksums(oracle):
    from fidibench_amd import Filter
    dims = (300, 257)
    rng = np.random.default_rng(4)
    f = rng.standard_normal(dims)
    flt = Filter(dims, [0.0, 0.0], [1.0, 1.0], {(0, 0): 0.6, (1, 0): 0.1, (0, -1): 0.3})
    flt.setInData(f)
    flt.applyFilter()
    out = flt.get_data("output").ravel(order="F")
    assert flt.computeCheckSum("output") == oracle.checksum(np.ascontiguousarray(out))
    assert flt.computeCheckSum("input") == oracle.checksum(
        np.ascontiguousarray(f.ravel(order="F")))
    flt.close()


# The sum of f[:at] is an odd multiple of u, and f[at] (in a chunk of its own
# from the sum's) lies next to half of u: the loop leaves the sum, a tie would
# move it to the even neighbour.
@pytest.mark.parametrize("sign", [1.0, -1.0])
@pytest.mark.parametrize("low", [1, 2])  # odd and even significands
@pytest.mark.parametrize("at", [2048, 5000, 65535])
def test_values_next_to_a_tie(oracle, sign, low, at):
    from fidibench_amd import Filter, Upwind
    half = 2.0 ** -53
    near = [half, np.nextafter(half, 0.0), np.nextafter(half, 1.0),
            3 * half, np.nextafter(3 * half, 0.0), np.nextafter(3 * half, 1.0)]
    for v in near + [-x for x in near]:
        f = np.zeros(65536)
        f[0], f[at] = sign * (1.5 + low * 2.0 ** -52), sign * v
        with Upwind((1.0,), (1.0,), (f.size,)) as up:
            up.set_field(f)
            assert up.checksum().hex() == oracle.checksum(f).hex(), (sign, low, at, v.hex())
            assert up.std().hex() == oracle.std(f).hex(), (sign, low, at, v.hex())
    flt = Filter((256, 256), [0.0, 0.0], [1.0, 1.0], {(0, 0): 1.0})
    flt.setInData(f)
    assert flt.computeCheckSum("input").hex() == oracle.checksum(f).hex()
    flt.close()


def test_values_next_to_a_tie_add_up(oracle):
    from fidibench_amd import Upwind
    f = np.zeros(65536)
    f[0] = 1.5 + 2.0 ** -52
    f[2048:4096:2], f[2049:4096:2] = -np.nextafter(2.0 ** -53, 0.0), 2.0 ** -52
    for g in (f, -f):
        with Upwind((1.0,), (1.0,), (g.size,)) as up:
            up.set_field(g)
            assert up.checksum().hex() == oracle.checksum(g).hex()


@pytest.mark.parametrize("n", [300 * 2048, 5000000])
def test_equal_values_drift_from_the_guess(oracle, n):
    """Sums that reach a power of two at a chunk's start."""
    from fidibench_amd import Upwind
    for x in (0.1, 8.0 / (3 * 2048), 8.0 / (77 * 2048), -1.0 / (5 * 2048)):
        f = np.full(n, x)
        with Upwind((1.0,), (1.0,), (n,)) as up:
            up.set_field(f)
            assert np.float64(up.checksum()).tobytes() == np.float64(oracle.checksum(f)).tobytes()


def test_checksums_of_one_filter_from_several_threads(oracle):
    """Each thread's folds share the filter's scratch."""
    import threading
    from fidibench_amd import Filter
    n = 300 * 2048 + 5
    f = np.random.default_rng(4).standard_normal(n)
    flt = Filter((n,), (0.0,), (1.0,), {(0,): 2.0, (1,): -0.5})
    flt.setInData(f)
    flt.applyFilter()
    want = {"input": oracle.checksum(f), "output": oracle.checksum(flt.get_data("output"))}
    wrong = []

    def fold(which):
        for _ in range(20):
            got = flt.computeCheckSum(which)
            if np.float64(got).tobytes() != np.float64(want[which]).tobytes():
                wrong.append((which, got))

    threads = [threading.Thread(target=fold, args=(w,)) for w in ("input", "output") * 2]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    flt.close()
    assert not wrong
