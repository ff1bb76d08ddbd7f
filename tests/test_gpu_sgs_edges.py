"""Inference kernel at the edges of its groups of two rows of 128 cells (a last row of its own, one cell
past a group, a last tile of one cell), both precisions, against the oracle.

Bounds: the median of an output 1e-4 and its largest error 2e-2 of the output's largest; both sides round
inputs and activations to bf16 from sums in another order (2^-8 of one of 64 terms)."""
import numpy as np
import pytest

import porturb_amd as pa
from oracle import oracle_py as o
from tests.helpers import random_state, small_config, WV, TKE, P1, P2
from tests.test_gpu_sgs import fine_state, model_for, rand_params, run_learned

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", [pa.PU_FP64, pa.PU_FP32], ids=["fp64", "fp32"])
@pytest.mark.parametrize("size", [(129, 7, 6), (128, 9, 5), (17, 5, 8), (255, 8, 5)], ids=str)
def test_inference_at_group_edges(size, precision):
    nx, ny, nz = size
    cfg = small_config(nx=nx, ny=ny, nz=nz, ord=5, tracers=[WV, TKE, P1, P2], dx=2., precision=precision)
    st, imm = random_state(cfg, seed=27, buildings=1, amp_u=1.0)
    print("case", size, precision, flush=True)
    P = rand_params(28, scale=0.1)
    om = np.array([0.02, 0, -0.01, 0.02, 0, 0.02, 0, 0, -1e-3], np.float32)
    os_ = np.array([0.01, 0.005, 0.005, 0.01, 0.005, 0.01, 1e-3, 1e-3, 1e-3], np.float32)
    gm, om_ = model_for(P, om, os_)
    _, tau, fl = run_learned(cfg, st, imm, gm, 0.02)
    rtau, rfl = o.les_apply_learned(cfg, st.copy(), imm, 0.02, om_)
    assert (fl == rfl).mean() >= 0.99
    for f in range(9):
        s = max(np.abs(rtau[f]).max(), 1e-30)
        err = np.abs(tau[f] - rtau[f])
        assert np.median(err) <= 1e-4 * s and err.max() <= 2e-2 * s, f
    gm.destroy()


@pytest.mark.parametrize("ratio,n", [(2, (17, 9, 5)), (3, (11, 7, 4)), (4, (13, 11, 3)), (6, (5, 3, 4))], ids=str)
def test_filter_ratios(ratio, n):
    """Box filter with one and with two threads a coarse cell, cells that do not fill a block.  Bounds as at
    ratio 2: 1e-12 of a field (sums of up to 216 terms in another order), 1e-6 of a float target."""
    nx, ny, nz = n
    cfg, st, imm = fine_state(ratio * nx, ratio * ny, ratio * nz)
    print("case", ratio, n, flush=True)
    cs = pa.CouplerState(cfg)
    cs.upload((st, imm))
    d = pa.Dycore(cfg)
    les, immc, tg = pa.sgs_filter(d.ctx, cs.c, cfg, ratio)
    r_les, r_imm, r_tg = o.sgs_filter(cfg, st, imm, ratio)
    assert np.array_equal(immc.download(np.float64, (nz + 2, ny + 2, nx + 2)), r_imm)
    g_les, g_tg = les.download(np.float64, (6, nz + 2, ny + 2, nx + 2)), tg.download(np.float32, (9, nz, ny, nx))
    for f in range(6):
        assert np.abs(g_les[f] - r_les[f]).max() <= 1e-12 * max(np.abs(r_les[f]).max(), 1e-30), f
    for f in range(9):
        assert np.abs(g_tg[f] - r_tg[f]).max() <= 1e-6 * max(np.abs(r_tg[f]).max(), 1e-30), f
