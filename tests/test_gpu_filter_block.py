"""Star stencils by the block kernel (radius 1 and 2, 2-D and 3-D) against
the oracle, bit for bit: tiles cut on each axis, last blocks of 1 plane to a
full one, grids narrower than a tile, both block sizes (the smaller one where
the grid has fewer than 256), and the sizes where the marching kernels with
cached stores and the streaming stores take over."""
from __future__ import annotations

import numpy as np
import pytest

from conftest import bits

pytestmark = pytest.mark.gpu


def _star(rng, nd, R):
    st = {tuple([0] * nd): float(rng.standard_normal())}
    for a in range(nd):
        for k in range(1, R + 1):
            for sg in (1, -1):
                o = [0] * nd
                o[a] = sg * k
                st[tuple(o)] = float(rng.standard_normal())
    return st


@pytest.mark.parametrize("R", [1, 2])
@pytest.mark.parametrize("dims", [
    (8, 8, 5), (31, 9, 6), (33, 17, 7), (3, 40, 9),          # small blocks
    (97, 49, 81), (160, 48, 82), (65, 95, 83), (160, 15, 400),  # 32 x 16 x 4
    (5, 6), (300, 7), (256, 1023),                           # 2-D, small blocks
    (257, 1025), (2, 2049), (513, 2050), (1000, 2055), (511, 2056)])      # 2-D, 8 rows
def test_block_kernel_bit_exact_vs_oracle(oracle, dims, R):
    from fidibench_amd import Filter
    nd = len(dims)
    rng = np.random.default_rng(sum(dims) + R)
    st = _star(rng, nd, R)
    ref = rng.standard_normal(int(np.prod(dims)))
    flt = Filter(dims, [0.0] * nd, [1.0] * nd, st)
    flt.setInData(ref)
    for it in range(2):
        flt.applyFilter()
        ref = oracle.filter_apply(ref, dims, list(st.items()))
        got = flt.get_data("output").ravel(order="F")
        assert np.array_equal(bits(got), bits(ref)), it
        flt.copyOutToIn()
    flt.close()


# 16 bytes a cell: below and above 160 MiB (3-D, radius 2) and 256 MiB
@pytest.mark.parametrize("dims,R", [((219, 217, 220), 2), ((221, 219, 218), 2),
                                    ((257, 256, 255), 1), ((257, 258, 256), 1),
                                    ((257, 258, 256), 2), ((4096, 4095), 2), ((4097, 4099), 2)])
def test_kernel_choice_by_size_bit_exact_vs_oracle(oracle, dims, R):
    from fidibench_amd import Filter
    nd = len(dims)
    rng = np.random.default_rng(R)
    st = _star(rng, nd, R)
    f0 = rng.standard_normal(int(np.prod(dims)))
    flt = Filter(dims, [0.0] * nd, [1.0] * nd, st)
    flt.setInData(f0)
    flt.applyFilter()
    ref = oracle.filter_apply(f0, dims, list(st.items()))
    assert np.array_equal(bits(flt.get_data("output").ravel(order="F")), bits(ref))
    flt.close()


# Planes of eight rows, radius 2: marched from 8 MiB (16 bytes a cell) and 128
# columns on, in blocks below.
@pytest.mark.parametrize("dims", [(127, 8, 530), (128, 8, 512), (128, 8, 513), (2000, 8, 33),
                                  (2001, 8, 40), (20000, 8, 6)])
def test_planes_of_eight_rows_bit_exact_vs_oracle(oracle, dims):
    test_block_kernel_bit_exact_vs_oracle(oracle, dims, 2)
