"""The relaxation kernel's branch-free bonded terms: every term is computed for every
pair of a node's four slots and weighted zero where the node lacks it, so nodes with
one to four neighbours, with and without a pi-vector, and each switch are where it can
go wrong.  One move, then the exact forces at the new geometry against the FP64 oracle
(max|dF| <= 1e-4 + 5e-6 max|F| eV/A, the bound of the other force tests).
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
SIZES = [5, 12, 40, 64, 65, 129, 250]
SWITCHES = [(dict(), (1, 1, 1, 1, 1)), (dict(Angles=-1), (1, 1, 1, 0, 1)), (dict(PiSigma=-1), (1, 1, 0, 1, 1)),
            (dict(PiPiI=-1), (1, 0, 1, 1, 1)), (dict(NonBonded=-1), (1, 1, 1, 1, 0))]


@pytest.mark.parametrize("switch,sw", SWITCHES)
def test_node_forces(orc, switch, sw):
    from firecore_amd import MMFF_multi as mm
    from firecore_amd import native
    mols = [native.gen_molecule(n, 300 + n, 0.1, n) for n in SIZES]
    native.set_opt(0.1, 0.02, 0.2, 1.1, 0.5, 0.8, 5)
    native.set_force_limit(0.0)
    native.init_systems(mols)
    print("case: node forces", switch, flush=True)
    mm.setSwitches_multi(**switch)
    try:
        native.relax(1, 1e-9, 0, False, True)
        B = native.Batch()
        for s, n in enumerate(SIZES):
            fo = orc.eval(dict(mols[s], apos=B.positions(s)), sw=sw)[0]
            d = np.abs(B.forces(s) - fo).max()
            assert d <= 1e-4 + 5e-6 * np.abs(fo).max(), (n, d, np.abs(fo).max())
    finally:
        mm.setSwitches_multi(NonBonded=1, Angles=1, PiSigma=1, PiPiI=1)
