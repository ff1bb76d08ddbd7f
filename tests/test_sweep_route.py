"""The choice between whole-line and segment kernels of the y and z sweeps (no device call), at grids whose two
kernels were timed (us per launch on an MI355X: lines, segments): it takes the faster one where they
are 6 % or more apart."""
import ctypes as C

import pytest

import porturb_amd as pa
from tests.helpers import small_config, WV, TKE, P1, P2

Z_TIMES = [
    # precision, order, nx, ny, nz, lines, segments
    ("fp32", 9, 256, 256, 33, 212.7, 242.0), ("fp32", 11, 256, 256, 33, 295.5, 339.1),
    ("fp32", 11, 300, 200, 100, 647.2, 705.5), ("fp32", 11, 148, 341, 66, 406.9, 443.4),
    ("fp32", 9, 410, 232, 34, 314.0, 372.1), ("fp32", 11, 410, 232, 34, 435.9, 536.9),
    ("fp32", 11, 307, 56, 38, 100.4, 115.3), ("fp32", 11, 265, 111, 65, 242.3, 265.0),
    ("fp32", 3, 500, 310, 90, 628.6, 483.7), ("fp32", 5, 500, 310, 90, 683.6, 601.0),
    ("fp32", 7, 500, 310, 90, 809.4, 754.6), ("fp32", 3, 124, 90, 40, 34.0, 31.2),
    ("fp64", 9, 256, 256, 33, 302.6, 360.5), ("fp64", 11, 256, 256, 33, 428.5, 506.8),
    ("fp64", 9, 300, 200, 100, 707.6, 759.2), ("fp64", 11, 300, 200, 100, 957.4, 1036.9),
    ("fp64", 9, 52, 460, 37, 141.6, 158.7), ("fp64", 3, 500, 310, 90, 776.6, 666.2),
    ("fp64", 5, 500, 310, 90, 958.8, 868.0), ("fp64", 7, 500, 310, 90, 1157.0, 1083.5),
    ("fp64", 5, 124, 90, 40, 58.9, 44.2), ("fp64", 7, 124, 90, 40, 65.7, 54.4),
    ("fp64", 9, 1024, 1024, 128, 14.1e3, 17.5e3),
]


def config(precision, ord_, nx, ny, nz, **kw):
    return small_config(nx=nx, ny=ny, nz=nz, ord=ord_, tracers=[WV, TKE, P1, P2],
                        precision=pa.PU_FP32 if precision == "fp32" else pa.PU_FP64, **kw)


@pytest.mark.parametrize("row", Z_TIMES, ids=lambda r: "%s-o%d-%dx%dx%d" % r[:5])
def test_z_takes_the_faster_kernel(row):
    assert pa.sweep_takes_segments(config(*row[:5]), 2) == (row[6] < row[5])


@pytest.mark.parametrize("ord_", (3, 5, 7, 9, 11))
def test_where_one_kernel_only_applies(ord_):
    for size in ((64, 64, 64), (24, 700, 60), (512, 256, 128)):
        assert not pa.sweep_takes_segments(config("fp32", ord_, *size), 1)
        for precision in ("fp32", "fp64"):
            assert pa.sweep_takes_segments(config(precision, ord_, *size, bc_y=pa.PU_BC_PRECURSOR), 1)
            assert pa.sweep_takes_segments(config(precision, ord_, *size, bc_z=pa.PU_BC_PERIODIC), 2)
    # columns whose offsets need more than 32 bits
    assert pa.sweep_takes_segments(config("fp64", ord_, 8192, 8192, 1024), 2)


def test_arguments():
    out = C.c_int()
    cfg = pa.to_pu_config(config("fp64", 5, 16, 16, 16))
    L = pa.lib()
    assert L.pu_sweep_route(C.byref(cfg), 1, None) == pa.PU_ERR_ARG
    assert L.pu_sweep_route(C.byref(cfg), 0, C.byref(out)) == pa.PU_ERR_ARG
    assert L.pu_sweep_route(C.byref(pa.to_pu_config(config("fp64", 4, 16, 16, 16))), 1, C.byref(out)) == pa.PU_ERR_UNSUPPORTED
