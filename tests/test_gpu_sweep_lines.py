"""Both kernels of the y and z sweeps at the edges of their tiles, each forced whatever the grid's size would
choose (PORTURB_SEGMENT_SWEEPS with PORTURB_SEGMENT_DIRS naming the directions of the segment kernel): lines of
one chunk of 32 cells, one cell more, two chunks and one cell, segments of 30 cells, lines of two cells.

FP64 against the oracle: 5e-11 of each field's largest tendency (the sums run in another order; see
test_gpu_sweep_edges.py).  Lines against segments: z bitwise in both precisions; y 1e-13 of a field's
largest in FP64 and 1e-5 in FP32, where the compiler fuses some multiply-adds differently."""
import os

import numpy as np
import pytest

import porturb_amd as pa
from oracle import oracle_py
from tests.helpers import random_state, small_config, WV, TKE, P1

pytestmark = pytest.mark.gpu


def tendencies(cfg, st, imm, dirs):
    os.environ["PORTURB_SEGMENT_SWEEPS"] = "1"
    os.environ["PORTURB_SEGMENT_DIRS"] = dirs
    try:
        cs = pa.CouplerState(cfg)
        cs.upload((st, imm))
        d = pa.Dycore(cfg)
    finally:
        del os.environ["PORTURB_SEGMENT_SWEEPS"], os.environ["PORTURB_SEGMENT_DIRS"]
    d.init(cs)
    return d.tendencies(cs)


def case(ord_, size, precision=pa.PU_FP64, **kw):
    nx, ny, nz = size
    cfg = small_config(nx=nx, ny=ny, nz=nz, ord=ord_, tracers=[WV, TKE, P1], precision=precision, **kw)
    print("case", ord_, size, precision, kw, flush=True)
    return (cfg,) + random_state(cfg, seed=51, buildings=2 if min(nx, ny) > 4 else 0)


def relative(t, ref):
    scale = np.maximum(np.abs(ref).reshape(ref.shape[0], -1).max(axis=1), 1e-300)
    return (np.abs(t - ref).reshape(ref.shape[0], -1).max(axis=1) / scale).max()


@pytest.mark.parametrize("dirs", ["", "yz"], ids=["lines", "segments"])
@pytest.mark.parametrize("size", [(9, 32, 33), (17, 33, 31), (8, 65, 64), (10, 29, 65), (7, 30, 30), (12, 61, 61)], ids=str)
@pytest.mark.parametrize("ord_", (3, 5, 7, 9, 11))
def test_each_kernel_against_oracle(ord_, size, dirs):
    cfg, st, imm = case(ord_, size)
    assert relative(tendencies(cfg, st, imm, dirs), oracle_py.Dycore(cfg, st, imm).tendencies(st)) < 5e-11


@pytest.mark.parametrize("precision", [pa.PU_FP64, pa.PU_FP32], ids=["fp64", "fp32"])
@pytest.mark.parametrize("size", [(40, 12, 70), (37, 10, 33), (24, 16, 64), (20, 12, 14), (16, 8, 129), (33, 61, 30)], ids=str)
@pytest.mark.parametrize("ord_", (3, 5, 7, 9, 11))
def test_z_kernels_agree_bitwise(ord_, size, precision):
    cfg, st, imm = case(ord_, size, precision)
    for y in ("", "y"):
        a, b = tendencies(cfg, st, imm, y), tendencies(cfg, st, imm, y + "z")
        assert np.abs(a).max() > 0 and np.array_equal(a, b), (y, relative(a, b))


@pytest.mark.parametrize("precision", [pa.PU_FP64, pa.PU_FP32], ids=["fp64", "fp32"])
@pytest.mark.parametrize("ord_,size,kw", [
    (9, (20, 70, 12), {}), (3, (16, 2, 10), {}), (3, (22, 2, 10), {}), (5, (24, 64, 10), {}), (5, (9, 33, 12), {}),
    (7, (16, 65, 10), dict(bc_z=pa.PU_BC_PERIODIC)), (9, (18, 20, 12), {}), (11, (11, 97, 12), {})], ids=str)
def test_y_kernels_agree(ord_, size, kw, precision):
    cfg, st, imm = case(ord_, size, precision, **kw)
    a, b = tendencies(cfg, st, imm, ""), tendencies(cfg, st, imm, "y")
    assert relative(a, b) < (1e-13 if precision == pa.PU_FP64 else 1e-5)
