"""The workspace of the absorbing-boundary step (grid_wf_propagate with ts_func set)."""
import os
import subprocess
import sys

import numpy as np
import pytest

import libgrid_amd as LG
from conftest import rel_l2

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.mark.parametrize("shape", [(16, 16, 8), (32, 16, 16), (16, 32, 8)])
def test_workspace_of_another_size_is_refused(shape):
    """A workspace that does not have the wavefunction's shape, smaller or of as many points, ends the call
    with the message of the copy that the step begins with, before any device is touched."""
    code = (
        "import libgrid_amd as LG; lib = LG.load();"
        "w = lib.grid_wf_alloc(16, 16, 16, 0.3, 1.0, LG.WF_PERIODIC_BOUNDARY, LG.WF_2ND_ORDER_FFT, b'w');"
        f"w.contents.cworkspace = lib.cgrid_alloc({shape[0]}, {shape[1]}, {shape[2]}, 0.3, None, None, b'work');"
        "v = lib.cgrid_alloc(16, 16, 16, 0.3, None, None, b'v');"
        "lib.grid_wf_boundary(w, None, 4, 11, 4, 11, 4, 11);"
        "lib.grid_wf_propagate(w, v, LG.c_complex.of(0.01))"
    )
    p = subprocess.run([sys.executable, "-c", code], capture_output=True, text=True, cwd=ROOT,
                       env=dict(os.environ, HIP_VISIBLE_DEVICES="", PYTHONPATH=ROOT))
    assert p.returncode != 0 and "Incompatible grids in cgrid_copy()" in p.stderr, p.stderr


def stepped(lg, psi, pot, prec, times, bounds=None, own=False):
    """(state, workspace) after steps of the given times; own: the wavefunction's grid is its workspace."""
    w = lg.grid_wf_alloc(*psi.shape, 0.3, 1.2, LG.WF_PERIODIC_BOUNDARY, LG.WF_2ND_ORDER_FFT, b"w")
    v = lg.cgrid_alloc(*psi.shape, 0.3, LG.boundary("cgrid_value_outside_periodic"), None, b"v")
    LG.set_cgrid(w.contents.grid, psi)
    LG.set_cgrid(v, pot)
    lg.cgrid_set_precision(w.contents.grid, prec)
    if bounds:
        lg.grid_wf_boundary(w, None, *bounds)
    if own:
        w.contents.cworkspace = w.contents.grid
    for t in times:
        lg.grid_wf_propagate(w, v, LG.c_complex.of(t))
    work = LG.get_cgrid(w.contents.cworkspace) if bounds else None
    out = LG.get_cgrid(w.contents.grid)
    if own:
        w.contents.cworkspace = None
    lg.cgrid_free(v)
    lg.grid_wf_free(w)
    return out, work


def inputs(shape):
    rng = np.random.default_rng(sum(shape))
    psi = (rng.standard_normal(shape) + 1j * rng.standard_normal(shape)) * 0.3 + 1.0
    return psi, rng.uniform(0, 1, shape) + 0.05j * rng.uniform(0, 1, shape), [b for n in shape for b in (n // 4, n - 1 - n // 4)]


@pytest.mark.gpu
@pytest.mark.parametrize("shape", [(16, 32, 24), (16, 8, 16)])
def test_grid_as_its_own_workspace(lg, shape):
    """Nothing is merged then: the real-time step and after it the imaginary-time one, in tile passes and
    in pencils.  The bar as in test_tile_pass.py: two steps' roundings, 2e-14."""
    psi, pot, bounds = inputs(shape)
    got, _ = stepped(lg, psi, pot, b"\x00", (0.02,), bounds, own=True)
    want, _ = stepped(lg, psi, pot, b"\x00", (0.02, -0.02j))
    assert rel_l2(got, want) < 2e-14


@pytest.mark.gpu
@pytest.mark.parametrize("prec,bar", [(b"\x00", 2e-14), (b"\x01", 1e-5)])
@pytest.mark.parametrize("shape", [(16, 32, 24), (48, 64, 16), (16, 8, 16), (1, 32, 16)])
def test_workspace_holds_the_imaginary_time_state(lg, shape, prec, bar):
    """After one step, and after two, the workspace reads as the imaginary-time step of the state that the
    last step began with, in tile passes and in pencils.  Bars of test_tile_pass.py."""
    psi, pot, bounds = inputs(shape)
    first, work = stepped(lg, psi, pot, prec, (0.02,), bounds)
    want, _ = stepped(lg, psi, pot, prec, (-0.02j,))
    assert rel_l2(work, want) < bar
    _, work = stepped(lg, psi, pot, prec, (0.02, 0.02), bounds)
    want, _ = stepped(lg, first, pot, prec, (-0.02j,))
    assert rel_l2(work, want) < bar
