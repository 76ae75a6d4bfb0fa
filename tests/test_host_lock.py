"""Grids locked to the host (host_lock) after device work."""
import numpy as np
import pytest

import libgrid_amd as LG
from conftest import rel_l2


@pytest.mark.gpu
@pytest.mark.parametrize("norm", (0, 1))
@pytest.mark.parametrize("shape", [(16, 16, 16), (16, 8, 64), (1, 32, 64)])
def test_values_of_a_locked_grid_can_be_read(lg, shape, norm):
    """A state that a step left transformed, with and without its normalisation outstanding, is read after
    the grid was locked as it is without the lock: the same kernels, so to the bit."""
    rng = np.random.default_rng(sum(shape))
    psi = rng.standard_normal(shape) + 1j * rng.standard_normal(shape)
    v = lg.rgrid_alloc(*shape, 0.3, LG.boundary("rgrid_value_outside_periodic"), None, b"v")
    LG.set_rgrid(v, rng.uniform(0, 1, shape))

    def run(lock):
        w = lg.grid_wf_alloc(*shape, 0.3, 1.2, LG.WF_PERIODIC_BOUNDARY, LG.WF_2ND_ORDER_FFT, b"w")
        LG.set_cgrid(w.contents.grid, psi)
        lg.grid_wf_gpe_propagate(w, v, 0.3, LG.c_complex.of(-0.05j), norm)
        w.contents.grid.contents.host_lock = lock
        out = LG.get_cgrid(w.contents.grid)
        lg.grid_wf_free(w)
        return out

    got, want = run(b"\x01"), run(b"\x00")
    lg.rgrid_free(v)
    assert np.array_equal(got, want) and rel_l2(got, psi) > 1e-3
