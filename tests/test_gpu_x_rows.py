"""x sweep at row lengths on either side of the choice between rows in waves of their own (a multiple of the 62
cells a wave owns, or up to two short of one) and rows laid end to end.

FP64 against the oracle, bound 5e-11 of each field's largest tendency (as for the other edges of the
sweeps' tiles).  FP32: a periodic flow repeated two and three times in x must have the tendencies of one
copy, at lengths that take the other layout; bound 1e-3 of a field's largest, which covers the limiter's
amplification of the last bits of the level means (a wrong neighbour is off by the tendency itself)."""
import numpy as np
import pytest

import porturb_amd as pa
from oracle import oracle_py
from tests.helpers import random_state, small_config, WV, TKE, P1

pytestmark = pytest.mark.gpu


def tendencies(cfg, st, imm):
    cs = pa.CouplerState(cfg)
    cs.upload((st, imm))
    d = pa.Dycore(cfg)
    d.init(cs)
    return d.tendencies(cs)


@pytest.mark.parametrize("bc_x", [pa.PU_BC_PERIODIC, pa.PU_BC_PRECURSOR], ids=["periodic", "open"])
@pytest.mark.parametrize("nx", [59, 60, 61, 62, 63, 122, 123, 124, 186])
@pytest.mark.parametrize("ord_", (3, 9, 11))
def test_row_layouts_against_oracle(ord_, nx, bc_x):
    cfg = small_config(nx=nx, ny=7, nz=13, ord=ord_, tracers=[WV, TKE, P1], bc_x=bc_x)
    st, imm = random_state(cfg, seed=41, buildings=2)
    print("case", ord_, nx, bc_x, flush=True)
    g = tendencies(cfg, st, imm)
    o = oracle_py.Dycore(cfg, st, imm).tendencies(st)
    scale = np.maximum(np.abs(o).reshape(o.shape[0], -1).max(axis=1), 1e-300)
    err = np.abs(g - o).reshape(g.shape[0], -1).max(axis=1) / scale
    assert err.max() < 5e-11, err


@pytest.mark.parametrize("nx", [31, 41, 61, 62])       # times 1, 2, 3: both layouts among them
@pytest.mark.parametrize("ord_", (3, 5, 7, 9, 11))
def test_repeated_flow_in_fp32(ord_, nx):
    cfg = small_config(nx=nx, ny=9, nz=13, ord=ord_, tracers=[WV, TKE, P1], precision=pa.PU_FP32)
    st, imm = random_state(cfg, seed=42, buildings=2)
    print("case", ord_, nx, flush=True)
    one = tendencies(cfg, st, imm)
    scale = np.maximum(np.abs(one).reshape(one.shape[0], -1).max(axis=1), 1e-300)[:, None, None, None]
    for m in (2, 3):
        wide = dict(cfg, nx=m * nx, xlen=m * cfg["xlen"])
        t = tendencies(wide, np.tile(st, (1, 1, 1, m)), np.tile(imm, (1, 1, m)))
        assert t.shape[-1] == m * nx
        for c in range(m):
            err = np.abs(t[..., c * nx:(c + 1) * nx] - one) / scale
            assert err.max() < 1e-3, (m, c, err.max())
