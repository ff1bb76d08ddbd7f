"""Sweeps at the edges of their tiles against the oracle: x rows around the 62 cells a wave owns, y
lines and z columns around the 32-cell chunks, periodic and open x, buildings beside the faces, flow
in both directions (the upwind cell of a face is read in opposite orders).

Bound: 5e-11 of each field's largest tendency.  Both sides evaluate the same sums in another order;
the oracle's smoothness indicators come from polynomial coefficients of the raw values, whose
rounding (1e-16 of the value, ~1e2 u for w and p) reaches a few 1e-11 of a tendency."""
import numpy as np
import pytest

import porturb_amd as pa
from oracle import oracle_py
from tests.helpers import random_state, small_config, WV, TKE, P1

pytestmark = pytest.mark.gpu

EDGES = [(61, 31, 32), (62, 32, 33), (63, 33, 31), (125, 65, 12), (11, 6, 64)]


@pytest.mark.parametrize("bc_x", [pa.PU_BC_PERIODIC, pa.PU_BC_PRECURSOR], ids=["periodic", "open"])
@pytest.mark.parametrize("size", EDGES, ids=str)
@pytest.mark.parametrize("ord_", (5, 9))
def test_sweeps_at_tile_edges(ord_, size, bc_x):
    nx, ny, nz = size
    cfg = small_config(nx=nx, ny=ny, nz=nz, ord=ord_, tracers=[WV, TKE, P1], bc_x=bc_x)
    st, imm = random_state(cfg, seed=31, buildings=2)
    print("case", ord_, size, bc_x, flush=True)
    cs = pa.CouplerState(cfg)
    cs.upload((st, imm))
    d = pa.Dycore(cfg)
    d.init(cs)
    g = d.tendencies(cs)
    o = oracle_py.Dycore(cfg, st, imm).tendencies(st)
    scale = np.maximum(np.abs(o).reshape(o.shape[0], -1).max(axis=1), 1e-300)
    err = np.abs(g - o).reshape(g.shape[0], -1).max(axis=1) / scale
    assert err.max() < 5e-11, err
