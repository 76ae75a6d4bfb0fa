"""Transforms of many contiguous rows, and where they go wrong if they do.

cgrid_fft runs one pass per axis, z, y and x, in place.  Undoing the outer axes of a wrong result's
difference one after the other in NumPy leaves it sparse at the pass that lost something, so a
failure names the pass, the elements and their values instead of one norm.

Bars as for test_row_pass.py: log2 N < 24 roundings in a row, each twice, 48 eps / 2 (FP64 1e-14); FP32
storage rounds the input and each of three passes, 4 * 6e-8, below 1e-6."""
import numpy as np
import pytest

import libgrid_amd as LG
from conftest import rel_l2


def stages(got, want):
    """(stage, elements off, [(index, difference)]) of a forward transform's result, last pass first."""
    diff, out = got - want, []
    for name, axis in (("after x", 0), ("after y", 1), ("after z", 2), ("input", None)):
        size = np.abs(diff)
        off = np.flatnonzero(size.ravel() > 1e-6 * np.linalg.norm(size))
        out.append((name, off.size, [(tuple(map(int, np.unravel_index(i, diff.shape))), complex(diff.ravel()[i])) for i in off[:16]]))
        if axis is not None:
            diff = np.fft.ifft(diff, axis=axis)
    return out


@pytest.mark.parametrize("stage,axes", [("after x", (2, 1, 0)), ("after y", (2, 1)), ("after z", (2,)), ("input", ())])
def test_a_lost_line_is_found(stage, axes):
    """Four neighbouring elements set to zero after a pass are reported there, and spread elsewhere."""
    rng = np.random.default_rng(5)
    a = rng.standard_normal((16, 12, 24)) + 1j * rng.standard_normal((16, 12, 24))
    want = np.fft.fftn(a)
    for ax in axes:
        a = np.fft.fft(a, axis=ax)
    a[3, 5, 8:12] = 0.0
    for ax in (2, 1, 0)[len(axes):]:
        a = np.fft.fft(a, axis=ax)
    found = {name: (n, at) for name, n, at in stages(a, want)}
    assert found[stage][0] == 4 and [i for i, _ in found[stage][1]] == [(3, 5, z) for z in range(8, 12)]
    assert min(n for n, _ in found.values()) == 4


@pytest.mark.gpu
@pytest.mark.parametrize("prec,bar", [(b"\x00", 1e-14), (b"\x02", 1e-6)])
@pytest.mark.parametrize("n", (96, 192, 384))
def test_many_rows(lg, n, prec, bar):
    """256 x 128 rows of a length with a factor 3 in FP64 arithmetic, each time in a new grid."""
    shape = (256, 128, n)
    rng = np.random.default_rng(n)
    a = rng.standard_normal(shape) + 1j * rng.standard_normal(shape)
    want = np.fft.fftn(a)
    for k in range(4):
        print(f"[case] {shape} precision {prec[0]} transform {k}", flush=True)
        g = lg.cgrid_alloc(*shape, 0.3, LG.boundary("cgrid_value_outside_periodic"), None, b"g")
        LG.set_cgrid(g, a)
        lg.cgrid_set_precision(g, prec)
        lg.cgrid_fft(g)
        got = LG.get_cgrid(g)
        lg.cgrid_free(g)
        err = rel_l2(got, want)
        assert err < bar, f"{shape} precision {prec[0]} transform {k}: {err:.2e}\n" + "\n".join(map(str, stages(got, want)))
