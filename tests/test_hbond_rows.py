"""Pair rows with H-bond charges in the relaxation kernel: the rows of H lie between those
of the other pair parameters and the reactions, and the proposal network's activations
are put over them.  Exact forces after two moves (in the learned form with the network
evaluated before each) against the FP64 oracle: max|dF| <= 1e-4 + 5e-6 max|F| eV/A, the
bound of the other force tests."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
SIZES = [4, 5, 6, 7, 40, 63, 64, 65, 127, 128, 129, 192, 193, 255, 256]


@pytest.mark.parametrize("form", ["plain", "constant", "learned"])
def test_forces_with_hbond_charges(orc, form):
    from firecore_amd import native
    mols = []
    for n in SIZES:
        m = native.gen_molecule(n, 700 + n, 0.05, n)
        m["REQs"][::3, 3] = -0.5
        m["REQs"][1::3, 3] = 0.4
        mols.append(m)
    native.set_opt(0.02, 0.005, 0.2, 1.1, 0.5, 0.8, 5)
    # forces come back clamped in the plain form, in the others those on pi-vectors
    native.set_force_limit(0.0 if form == "plain" else 1.0)
    try:
        if form == "learned":
            native.set_proposal_weights(np.load("firecore_amd/proposal_weights.npy"))
            native.set_proposal_every(1)
            native.set_precond(2, 3.0, 127.0)
        elif form == "constant":
            native.set_precond(1, 2.0, 127.0)
        native.init_systems(mols)
        print("case: H-bond rows", form, flush=True)
        native.relax(2, 1e-9, 0, False, True)
        B = native.Batch()
        assert (np.array(B.nsteps) == 2).all()
        for s, n in enumerate(SIZES):
            fo = orc.eval(dict(mols[s], apos=B.positions(s)))[0]
            rows = slice(None if form == "plain" else n)
            d = np.abs(B.forces(s)[rows] - fo[rows]).max()
            assert d <= 1e-4 + 5e-6 * np.abs(fo).max(), (n, d, np.abs(fo).max())
    finally:
        native.set_precond(0)
        native.set_proposal_every(128)
