"""Closure update at the edges of its 16 x 4 x 4 tiles: one short, exact and one over in each direction,
periodic and precursor x, buildings, two diffused tracers, against the oracle.

Bounds: FP64 1e-12 of each field's norm, the closure's bound elsewhere; FP32 mode 1e-4 of the largest
increment (float rounding of the box values and fluxes, 1e-6 relative, cancelled to ~1e-2 of themselves
in a divergence)."""
import numpy as np
import pytest

import porturb_amd as pa
from oracle import oracle_py
from tests.helpers import random_state, rel_norms, small_config, WV, TKE, P1, P2

pytestmark = pytest.mark.gpu

EDGES = [(15, 4, 9), (16, 5, 8), (17, 7, 12), (33, 8, 11), (31, 9, 5)]


@pytest.mark.parametrize("precision", [pa.PU_FP64, pa.PU_FP32], ids=["fp64", "fp32"])
@pytest.mark.parametrize("bc_x", [pa.PU_BC_PERIODIC, pa.PU_BC_PRECURSOR], ids=["periodic", "open"])
@pytest.mark.parametrize("size", EDGES, ids=str)
def test_update_at_tile_edges(size, bc_x, precision):
    nx, ny, nz = size
    cfg = small_config(nx=nx, ny=ny, nz=nz, ord=3, tracers=[WV, TKE, P1, P2], bc_x=bc_x, precision=precision)
    st, imm = random_state(cfg, seed=12, buildings=2)
    print("case", size, bc_x, precision, flush=True)
    cs = pa.CouplerState(cfg)
    cs.upload((st, imm))
    d = pa.Dycore(cfg)
    d.init(cs)
    d.les_apply(cs, 0.3)
    g = cs.download()
    ref = st.copy()
    oracle_py.les_apply(cfg, ref, imm, 0.3)
    if precision == pa.PU_FP64:
        assert rel_norms(g, ref).max() < 1e-12
    else:
        for f in range(1, g.shape[0]):
            inc_r, inc_g = ref[f] - st[f], g[f] - st[f]
            assert np.abs(inc_g - inc_r).max() <= 1e-4 * max(np.abs(inc_r).max(), 1e-300), f
