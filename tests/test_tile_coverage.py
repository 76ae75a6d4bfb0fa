"""Every instantiation of the tile passes that a plan can choose has run against the oracle: an A-pass is
built for (precision, z points, rows), a B-pass for (precision, x points, h points)."""
import ctypes as C

import pytest

import libgrid_amd as LG
from test_tile_pass import LENGTHS, LONG, steps

ALL = (16, 24, 32, 48, 64, 96, 128, 192, 256, 384, 512)
# 512 points are split into 64 rows in FP64 only beside an x of more than 256 points or with a factor 3
ROWS64 = [(24, 512, n) for n in (24, 32, 48, 64, 96, 128, 192)]
TESTED = [(n, n1, 16) for n1 in LENGTHS for n in LENGTHS] + [(16, n1, n) for n1 in LENGTHS for n in LENGTHS] + LONG + ROWS64
TESTED += [(1, n1, n2) for n1 in (64, 96, 128, 192, 256, 384, 512, 1024) for n2 in (32, 48, 64, 96, 384, 512) if n2 != 48 or n1 >= 128]


class Tile(C.Structure):
    """The part of hgrid_tile that a plan fills in; the rest as bytes."""
    _fields_ = [("psi", C.c_void_p), ("out", C.c_void_p), ("prec", C.c_int), ("n0", C.c_long), ("n1", C.c_long), ("n2", C.c_long),
                ("flat", C.c_int), ("rows", C.c_int), ("nh", C.c_int), ("rest", C.c_char * 1024)]


def instances(prec, shape):
    lib = LG.load()
    lib.hgrid_tile_plan.restype = C.c_int
    lib.hgrid_tile_plan.argtypes = [C.c_int, C.c_long, C.c_long, C.c_long, C.c_void_p]
    t = Tile()
    if not lib.hgrid_tile_plan(prec, *shape, C.byref(t)):
        return set()
    return {("A", prec, t.n2, t.rows), ("B", prec, t.nh if t.flat else t.n0, 1 if t.flat else t.nh)}


def test_every_planned_instance_is_among_the_tested_shapes():
    shapes = [(a, b, c) for a in ALL for b in ALL for c in ALL] + [(1, b, c) for b in ALL + (1024,) for c in ALL]
    for prec in (LG.HGRID_C128, LG.HGRID_C64):
        planned = set().union(*(instances(prec, s) for s in shapes))
        tested = set().union(*(instances(prec, s) for s in TESTED))
        assert len(planned) > 80 and planned == tested, planned ^ tested


@pytest.mark.gpu
@pytest.mark.parametrize("shape", ROWS64)
def test_64_rows_of_every_length(lg, orc, shape):
    """Steps of every kind, bars of test_tile_pass.py."""
    for what, err, bar in steps(lg, orc, shape):
        assert err < bar, f"{shape} {what}: rel L2 {err:.3e}"
