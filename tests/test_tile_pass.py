"""Tile passes (csrc/hip/tile_pass.hpp): the shapes they take, and steps on every tile geometry
against the oracle.

Bars of the GPU steps, fixed by the number of roundings: two steps are 8 transforms of at most 2^22
points, each about log2 N roundings in a row, 8 * 22 * eps / 2 with eps = 1.1e-16 or 6e-8 in the
worst case of all rounding the same way; 2e-14 and 1e-5.  A wrong index, twiddle or factor is of
order 1."""
import ctypes as C

import numpy as np
import pytest

import libgrid_amd as LG
from conftest import rel_l2

LENGTHS = (16, 24, 32, 48, 64, 96, 128, 192, 256)
BARS = {b"\x00": 2e-14, b"\x01": 1e-5}


def planned(prec, n0, n1, n2):
    lib = LG.load()
    lib.hgrid_tile_plan.restype = C.c_int
    lib.hgrid_tile_plan.argtypes = [C.c_int, C.c_long, C.c_long, C.c_long, C.c_void_p]
    return bool(lib.hgrid_tile_plan(prec, n0, n1, n2, C.create_string_buffer(1024)))


def test_shapes_taken_and_left():
    for n in LENGTHS[2:]:
        for prec in (LG.HGRID_C128, LG.HGRID_C64):
            assert planned(prec, n, n, n), (prec, n)
        assert not planned(LG.HGRID_C64X, n, n, n)  # FP32 storage with FP64 arithmetic
    assert planned(LG.HGRID_C128, 1, 384, 512) and planned(LG.HGRID_C64, 1, 1024, 64)
    for shape in ((64, 64, 512), (512, 64, 64), (64, 512, 64), (384, 256, 512)):
        assert planned(LG.HGRID_C128, *shape) and planned(LG.HGRID_C64, *shape), shape
    # one tile would be 2^15 FP64 values, twice what a CU's registers hold; in FP32 pencils are faster
    assert not planned(LG.HGRID_C128, 512, 512, 512) and not planned(LG.HGRID_C64, 512, 512, 512)
    assert planned(LG.HGRID_C64, 64, 512, 512) and planned(LG.HGRID_C64, 384, 384, 384)
    for shape in ((8, 64, 64), (64, 12, 64), (1, 1, 64), (1, 32, 64), (64, 1024, 64), (64, 64, 1024), (1, 64, 24)):
        assert not planned(LG.HGRID_C128, *shape), shape


def steps(lg, orc, shape):
    """Errors of two steps of each kind: imaginary and real time with a real potential (with and
    without the density), real time with a complex one (plain, with cutoff, 4th order)."""
    rng = np.random.default_rng(sum(shape))
    step, mass = 0.3, 1.2
    psi = (rng.standard_normal(shape) + 1j * rng.standard_normal(shape)) * 0.3 + 1.0
    psi /= np.sqrt(np.sum(np.abs(psi) ** 2) * step ** sum(n > 1 for n in shape))
    v = rng.uniform(0, 1, shape)
    pot = (v + 0.05j * rng.uniform(0, 1, shape)).astype(np.complex128)
    kmax = 0.6 * np.sqrt(sum((np.pi / step) ** 2 for n in shape if n > 1))
    k0 = (0.2, -0.1, 0.3)

    def run(prec, prop, one):
        w = lg.grid_wf_alloc(*shape, step, mass, LG.WF_PERIODIC_BOUNDARY, prop, b"w")
        w.contents.kmax = kmax
        LG.set_cgrid(w.contents.grid, psi)
        lg.cgrid_set_momentum(w.contents.grid, *k0)
        lg.cgrid_set_precision(w.contents.grid, prec)
        for _ in range(2):
            one(w)
        out = LG.get_cgrid(w.contents.grid)
        lg.grid_wf_free(w)
        return out

    vr = lg.rgrid_alloc(*shape, step, LG.boundary("rgrid_value_outside_periodic"), None, b"v")
    LG.set_rgrid(vr, v)
    vp = lg.cgrid_alloc(*shape, step, LG.boundary("cgrid_value_outside_periodic"), None, b"pot")
    LG.set_cgrid(vp, pot)
    for g, time, norm in ((0.3, -0.05j, 1), (0.0, -0.05j, 1), (0.3, 0.03, 0), (0.3, 0.03 - 0.02j, 0)):
        ref = psi.copy()
        for _ in range(2):
            orc.gpe_step_inplace(ref, v, g, step, mass, k0, time, normalize=bool(norm))
        for prec, bar in BARS.items():
            got = run(prec, LG.WF_2ND_ORDER_FFT, lambda w: lg.grid_wf_gpe_propagate(w, vr, g, LG.c_complex.of(time), norm))
            yield f"gpe g {g} t {time} precision {prec[0]}", rel_l2(got, ref), bar
    for prop, name in ((LG.WF_2ND_ORDER_FFT, ""), (LG.WF_2ND_ORDER_CFFT, "cfft_"), (LG.WF_4TH_ORDER_FFT, "4th_")):
        ref = psi.copy()
        for _ in range(2):
            getattr(orc, f"wf_propagate_{name}inplace")(ref, pot, step, mass, k0, 0.02, *([kmax] if "cfft" in name else []))
        for prec, bar in BARS.items():
            got = run(prec, prop, lambda w: lg.grid_wf_propagate(w, vp, LG.c_complex.of(0.02)))
            yield f"propagate {name} precision {prec[0]}", rel_l2(got, ref), bar
    if min(shape) > 1:  # absorbing boundary: two such steps of either time a step, and their merge
        bounds = [b for n in shape for b in (n // 4, n - 1 - n // 4)]
        ref = psi.copy()
        for _ in range(2):
            orc.wf_propagate_absorb_inplace(ref, pot, step, mass, k0, 0.02, tuple(bounds), None)

        def absorbed(w):
            lg.grid_wf_boundary(w, None, *bounds)
            lg.grid_wf_propagate(w, vp, LG.c_complex.of(0.02))

        for prec, bar in BARS.items():
            yield f"absorbing precision {prec[0]}", rel_l2(run(prec, LG.WF_2ND_ORDER_FFT, absorbed), ref), 2 * bar
    lg.cgrid_free(vp)
    lg.rgrid_free(vr)


@pytest.mark.gpu
@pytest.mark.parametrize("n1", LENGTHS)
@pytest.mark.parametrize("axis", ["x", "z"])
def test_every_tile_geometry(lg, orc, axis, n1):
    """Every (x, h) geometry of the B-pass and every (z, rows) geometry of the A-pass."""
    for n in LENGTHS:
        shape = (n, n1, 16) if axis == "x" else (16, n1, n)
        print(f"[case] {shape}", flush=True)
        for what, err, bar in steps(lg, orc, shape):
            assert err < bar, f"{shape} {what}: rel L2 {err:.3e}"


LONG = [(n, n1, 16) for n in (384, 512) for n1 in (16, 48, 96, 128, 192, 256, 384, 512)]
LONG += [(16, n1, n) for n in (384, 512) for n1 in (16, 32, 64, 256, 384, 512)]
LONG += [(n, n1, 32) for n in (16, 256) for n1 in (384, 512)] + [(16, 512, n) for n in LENGTHS] + [(24, 512, 256)]


@pytest.mark.gpu
@pytest.mark.parametrize("shape", LONG)
def test_long_axes(lg, orc, shape):
    """Axes of 384 and 512 points: the same, and every z with the 64 rows of the longest middle axes."""
    for what, err, bar in steps(lg, orc, shape):
        assert err < bar, f"{shape} {what}: rel L2 {err:.3e}"


@pytest.mark.gpu
@pytest.mark.parametrize("n1", (64, 96, 128, 192, 256, 384, 512, 768, 1024))
def test_every_2d_geometry(lg, orc, n1):
    for n2 in (32, 48, 64, 96, 384, 512):
        for shape in ((1, n1, n2), (n1, 1, n2)):
            if n1 == 768 or (n2 == 48 and n1 < 128):  # 768 is no FFT length
                continue
            print(f"[case] {shape}", flush=True)
            for what, err, bar in steps(lg, orc, shape):
                assert err < bar, f"{shape} {what}: rel L2 {err:.3e}"


@pytest.mark.gpu
@pytest.mark.parametrize("prec", sorted(BARS))
@pytest.mark.parametrize("shape", [(16, 16, 16), (32, 96, 48), (1, 96, 64), (16, 8, 64), (1, 32, 64)])
def test_copy_between_steps(lg, shape, prec):
    """A copy of a state between fused steps, in tile form or a pencil's deferred form and with its
    normalisation outstanding, holds the values that the grid then shows, and the next step goes on
    as if there had been no copy: the same kernels on the same values, so to the bit."""
    rng = np.random.default_rng(sum(shape))
    psi = rng.standard_normal(shape) + 1j * rng.standard_normal(shape)
    v = lg.rgrid_alloc(*shape, 0.3, LG.boundary("rgrid_value_outside_periodic"), None, b"v")
    LG.set_rgrid(v, rng.uniform(0, 1, shape))

    def run(copied):
        w = lg.grid_wf_alloc(*shape, 0.3, 1.2, LG.WF_PERIODIC_BOUNDARY, LG.WF_2ND_ORDER_FFT, b"w")
        out = lg.cgrid_alloc(*shape, 0.3, LG.boundary("cgrid_value_outside_periodic"), None, b"out")
        LG.set_cgrid(w.contents.grid, psi)
        lg.cgrid_set_precision(w.contents.grid, prec)
        lg.cgrid_set_precision(out, prec)
        copies = []
        for i in range(3):
            lg.grid_wf_gpe_propagate(w, v, 0.3, LG.c_complex.of(-0.05j), 1)
            if copied:
                lg.cgrid_copy(out, w.contents.grid)
                copies.append(LG.get_cgrid(out))
        end = LG.get_cgrid(w.contents.grid)
        lg.cgrid_free(out)
        lg.grid_wf_free(w)
        return end, copies

    plain, _ = run(False)
    end, copies = run(True)
    lg.rgrid_free(v)
    assert np.array_equal(end, plain)
    assert np.array_equal(copies[-1], end)
    norm = np.sum(np.abs(copies[0]) ** 2) * 0.3 ** sum(n > 1 for n in shape)
    assert abs(norm - 1.0) < 1e-12 + (1e-6 if prec == b"\x01" else 0.0)
