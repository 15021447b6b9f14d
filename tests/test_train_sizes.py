"""The training kernels' splits over waves: 16-row blocks shared by pairs of waves, the
head's sum over quarters of the atoms, the mean over every 16th system.  Gradients of
batches of 1, 15, 16, 17 and 33 systems of one size at the edges of those splits against
the oracle's backward pass (relative L2 norm per parameter block < 2e-2, the bound of the
BF16 gradients in the other tests)."""
import numpy as np
import pytest

from firecore_amd import native
from oracle import mlp
from test_proposal import _setup_batch, _systems

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nsys,natoms", [(1, 16), (15, 17), (16, 31), (17, 4), (33, 33), (2, 255), (2, 256)])
def test_gradient_at_edge_sizes(nsys, natoms):
    rng = np.random.default_rng(nsys)
    print("case: training gradient", nsys, natoms, flush=True)
    th = _setup_batch(nsys, 9900, natoms, natoms)
    try:
        out, feats = native.proposal_forward()
        B = native.Batch()
        dout = rng.normal(size=out.shape).astype(np.float32)
        g_dev = native.proposal_backward(dout).astype(np.float64)
        g_ref = np.zeros(mlp.NPARAM)
        for s, N, M, a0, n0, v0 in _systems(B):
            nb = mlp.neighbour_lists(N, B.neighs[a0:a0 + N])
            _, cache = mlp.forward(th, feats[a0:a0 + N].astype(np.float64), nb, bf=True)
            g_ref += mlp.backward(th, cache, dout[a0:a0 + N].astype(np.float64), nb, bf=True)
        g_ref /= B.nsys
        o = 0
        for name, sh in mlp.PARAM_SHAPES:
            n = int(np.prod(sh))
            a, b = g_dev[o:o + n], g_ref[o:o + n]
            rel = np.linalg.norm(a - b) / (np.linalg.norm(b) + 1e-12)
            assert rel < 2e-2, (name, rel)
            o += n
    finally:
        native.set_precond(0)
