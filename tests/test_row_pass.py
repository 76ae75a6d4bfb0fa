"""Plain transforms of contiguous rows (csrc/hip/row_pass.hpp) against NumPy's in 64 bits.

Bars, fixed by the number of roundings: a transform of N points rounds about log2 N <= 24 times in a
row, each time twice (twiddle and butterfly), all the same way in the worst case: 48 eps / 2 with
eps = 2.2e-16 or 1.2e-7, 1e-14 and 5e-6; FP32 storage with FP64 arithmetic rounds the input and
after each of three passes, 4 * 6e-8, below 1e-6."""
import numpy as np
import pytest

import libgrid_amd as LG
from conftest import rel_l2

BARS = {b"\x00": 1e-14, b"\x01": 5e-6, b"\x02": 1e-6}


@pytest.mark.gpu
@pytest.mark.parametrize("n", (64, 96, 128, 192, 256, 384, 512))
@pytest.mark.parametrize("rows", [(1, 2), (2, 3), (16, 6), (256, 128)])
def test_rows_of_every_length(lg, rows, n):
    """One row or two in a workgroup's tile, tiles cut off by the end, and (the last) the larger
    workgroups, whose last tile is cut off where three divides the length."""
    shape = (*rows, n)
    rng = np.random.default_rng(n)
    a = rng.standard_normal(shape) + 1j * rng.standard_normal(shape)
    want = np.fft.fftn(a)
    for prec, bar in BARS.items():
        print(f"[case] {shape} precision {prec[0]}", flush=True)
        g = lg.cgrid_alloc(*shape, 0.3, LG.boundary("cgrid_value_outside_periodic"), None, b"g")
        LG.set_cgrid(g, a)
        lg.cgrid_set_precision(g, prec)
        lg.cgrid_fft(g)
        err = rel_l2(LG.get_cgrid(g), want)
        lg.cgrid_inverse_fft_norm(g)
        back = rel_l2(LG.get_cgrid(g), a)
        lg.cgrid_free(g)
        assert err < bar and back < 2 * bar, f"{shape} precision {prec[0]}: {err:.2e} {back:.2e}"
