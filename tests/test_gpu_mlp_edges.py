"""Training kernel at the edges of its 64-sample blocks and of the reduction's 32-block batches, rows
gathered through an index list, against the oracle.

Bound: 2e-2 of the gradient's norm and of the loss.  Both sides round activations and their gradients
to bf16 from sums in another order; a rounding that falls the other way moves one of them by 2^-8, and
a single sample has few others to average it."""
import numpy as np
import pytest

import porturb_amd as pa
from oracle import oracle_py as o
from tests.test_gpu_sgs import rand_params

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", (1, 63, 64, 65, 2048, 2049, 4100))
def test_gradient_at_block_edges(n):
    print("case", n, flush=True)
    P = rand_params(41)
    rng = np.random.default_rng(n)
    X = rng.standard_normal((n + 50, pa.SGS_NIN)).astype(np.float32)
    T = rng.standard_normal((n + 50, pa.SGS_NOUT)).astype(np.float32)
    rows = rng.permutation(n + 50)[:n].astype(np.int32)
    dT, dI = pa.DeviceBuffer(T.nbytes), pa.DeviceBuffer(rows.nbytes)
    dT.upload(T)
    dI.upload(rows)
    m = pa.Mlp(P)
    loss, G = m.loss_grad(pa.pack_inputs(X), dT, n, idx=dI)
    lref, Gref = o.mlp_loss_grad(P, X[rows], T[rows], bf16=True)
    assert abs(loss - lref) <= 2e-2 * lref
    assert np.linalg.norm(G - Gref) <= 2e-2 * np.linalg.norm(Gref)
    m.destroy()
