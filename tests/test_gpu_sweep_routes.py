"""The y and z sweeps choose between whole lines and segments by the grid's size.  At sizes on either side
of that choice, the chosen route against both kernels by themselves (PORTURB_SEGMENT_SWEEPS with
PORTURB_SEGMENT_DIRS naming the directions of the segment kernel, the others by lines), periodic and open
x, both precisions, one cell and one chunk more or less.

Bounds: z bitwise.  y in FP64 1e-13 of each tendency's largest (the same sums, multiply-adds fused
differently); in FP32 the route is always the line kernel, so its bits."""
import os

import numpy as np
import pytest

import porturb_amd as pa
from tests.helpers import random_state, small_config, WV, TKE, P1

pytestmark = pytest.mark.gpu

SIZES = [(48, 40, 32), (9, 31, 33), (8, 30, 128), (33, 61, 30), (130, 8, 65), (64, 64, 64)]


def tendencies(cfg, st, imm, dirs):
    if dirs is not None:
        os.environ["PORTURB_SEGMENT_SWEEPS"] = "1"
        os.environ["PORTURB_SEGMENT_DIRS"] = dirs
    try:
        cs = pa.CouplerState(cfg)
        cs.upload((st, imm))
        d = pa.Dycore(cfg)
    finally:
        os.environ.pop("PORTURB_SEGMENT_SWEEPS", None)
        os.environ.pop("PORTURB_SEGMENT_DIRS", None)
    d.init(cs)
    return d.tendencies(cs)


@pytest.mark.parametrize("precision", [pa.PU_FP64, pa.PU_FP32], ids=["fp64", "fp32"])
@pytest.mark.parametrize("ord_,bc_x", [(5, pa.PU_BC_PERIODIC), (9, pa.PU_BC_PRECURSOR)])
@pytest.mark.parametrize("size", SIZES, ids=str)
def test_chosen_route_matches_both_kernels(size, ord_, bc_x, precision):
    nx, ny, nz = size
    cfg = small_config(nx=nx, ny=ny, nz=nz, ord=ord_, tracers=[WV, TKE, P1], bc_x=bc_x, precision=precision)
    st, imm = random_state(cfg, seed=17, buildings=2)
    print("case", size, ord_, bc_x, precision, flush=True)
    chosen = tendencies(cfg, st, imm, None)
    scale = np.maximum(np.abs(chosen).reshape(chosen.shape[0], -1).max(axis=1), 1e-300)
    for dirs in ("", "z", "y", "yz"):
        t = tendencies(cfg, st, imm, dirs)
        err = np.abs(t - chosen).reshape(t.shape[0], -1).max(axis=1) / scale
        if precision == pa.PU_FP32 and "y" not in dirs:
            assert np.array_equal(t, chosen), (dirs, err)
        else:
            assert err.max() <= (1e-13 if precision == pa.PU_FP64 else 1e-5), (dirs, err)
