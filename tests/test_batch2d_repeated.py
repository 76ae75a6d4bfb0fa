"""One wavefunction given for several problems of a batched relaxation."""
import ctypes as C

import numpy as np
import pytest

import libgrid_amd as LG


@pytest.mark.gpu
def test_a_repeated_wavefunction_keeps_its_last_problem(lg):
    """32 problems of 256 x 256 points, two wavefunctions taking turns: each ends with the state of the
    last problem it was given for, to the bit as with wavefunctions of its own (every problem runs by
    itself, its sums in a fixed order), and every problem reports its own energy."""
    n, ns = 256, 32
    rng = np.random.default_rng(11)
    psi = np.exp(-((np.arange(n) - 128.0) ** 2) / 800.0)
    psi = (psi[:, None] * psi[None, :]).reshape(1, n, n).astype(np.complex128)
    pots = []
    for _ in range(ns):
        r = lg.rgrid_alloc(1, n, n, 0.2, LG.boundary("rgrid_value_outside_periodic"), None, b"v")
        LG.set_rgrid(r, rng.uniform(0, 1, (1, n, n)))
        pots.append(r)

    def relax(distinct):
        own = []
        for _ in range(distinct):
            w = lg.grid_wf_alloc(1, n, n, 0.2, 1.0, LG.WF_PERIODIC_BOUNDARY, LG.WF_2ND_ORDER_FFT, b"w")
            LG.set_cgrid(w.contents.grid, psi)
            own.append(w)
        e, st = (C.c_double * ns)(), (C.c_long * ns)()
        lg.grid_wf_batch2d_relax(ns, (LG.WF * ns)(*(own[i % distinct] for i in range(ns))), (LG.RG * ns)(*pots), 0.1, 1e-30, 16, e, st)
        out = [LG.get_cgrid(w.contents.grid) for w in own]
        for w in own:
            lg.grid_wf_free(w)
        return out, list(e)

    want, energies = relax(ns)
    got, repeated = relax(2)
    for r in pots:
        lg.rgrid_free(r)
    assert repeated == energies and len(set(energies)) == ns
    assert np.array_equal(got[0], want[ns - 2]) and np.array_equal(got[1], want[ns - 1])
