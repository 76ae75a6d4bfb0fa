"""The 256^3 FP64 step runs in tile passes: the benchmark's roofline line takes their HBM traffic from
the committed rocprofv3 summary, so each must be found there under the instantiation that the library
is built with and plans for, with the pass's algorithmic bytes: the A-pass moves whole lines (1 %, as
for the pencils); of the B-passes two workgroups share each 128-byte line, and what their
common L2 has dropped in between is moved twice (6 %)."""
import ctypes as C
import os

import pytest

import bench
import libgrid_amd as LG
from test_tile_coverage import Tile

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.mark.parametrize("name,excess", [("tile_kin", 0.01), ("tile_gpe", 0.06), ("tile_pre", 0.06)])
def test_traffic_found_and_algorithmic(name, excess):
    traffic = bench.profiled_traffic(name, 256)
    assert traffic is not None, f"{name}: no line for {bench.TILE_SYMBOL[name]} in the traffic summary"
    assert abs(traffic / (bench.pass_bytes_per_point(name, 16) * 256**3) - 1.0) < excess


def test_statistics_and_library_name_every_pass():
    text = open(os.path.join(ROOT, "profiles", "gpe256_tile_kernel_stats.txt")).read()
    built = open(LG.load()._name, "rb").read()
    for name, sym in bench.TILE_SYMBOL.items():
        assert sym in text, name
        kernel, args = sym.rstrip(">").split("<", 1)
        last = args.split(", ")[-1]
        mangled = f"{kernel}I15HIP_vector_typeIdLj2EELi256ELi16EL" + ("b1" if last == "true" else f"i{last}") + "EE"
        assert mangled.encode() in built, mangled
    lib = LG.load()
    lib.hgrid_tile_plan.restype = C.c_int
    lib.hgrid_tile_plan.argtypes = [C.c_int, C.c_long, C.c_long, C.c_long, C.c_void_p]
    t = Tile()
    assert lib.hgrid_tile_plan(LG.HGRID_C128, 256, 256, 256, C.byref(t)) and (t.rows, t.nh) == (16, 16)
