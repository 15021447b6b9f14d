"""The persistent kernel's pair loop over periodic rows: offsets are taken four
at a time and the exclusion word of the last offset is kept in a register, so
sizes around multiples of 4, 32 and 64 offsets and of 64 atoms are where it can
go wrong.  One move, then the exact forces at the new geometry against the FP64
oracle (max|dF| <= 1e-4 + 5e-6 max|F| eV/A, the bound of the other force tests),
without and with H-bond charges (another layout of the rows)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
SIZES = [4, 5, 6, 7, 8, 9, 15, 16, 17, 62, 63, 64, 65, 66, 126, 127, 128, 129, 130, 190, 192, 193, 254, 255, 256]


@pytest.mark.parametrize("hbond", [False, True])
def test_pair_forces_at_edge_sizes(orc, hbond):
    from firecore_amd import native
    mols = [native.gen_molecule(n, 700 + n, 0.02, n) for n in SIZES]
    if hbond:
        for m in mols:
            m["REQs"] = np.array(m["REQs"])
            m["REQs"][0::3, 3] = -0.5
            m["REQs"][1::3, 3] = 0.4
    native.set_opt(0.1, 0.02, 0.2, 1.1, 0.5, 0.8, 5)
    native.set_force_limit(0.0)
    native.init_systems(mols)
    print("case: pair rows, hbond=%s" % hbond, flush=True)
    native.relax(1, 1e-9, 0, False, True)
    B = native.Batch()
    for s, n in enumerate(SIZES):
        fo = orc.eval(dict(mols[s], apos=B.positions(s)))[0]
        d = np.abs(B.forces(s) - fo).max()
        assert d <= 1e-4 + 5e-6 * np.abs(fo).max(), (n, d, np.abs(fo).max())
