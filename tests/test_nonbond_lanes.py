"""The wave-per-atom non-bonded kernel (batches with periodic molecules or substrate
atoms): lanes take every 64th (atom, image) pair, so 1, 63..65 and more images, molecules
of fewer atoms than a workgroup's waves, a vacuum molecule in the same batch, and a
substrate of few and of many terms are where it can go wrong.  Device forces and energies
against the FP64 oracle (max|dF| <= 1e-4 + 5e-6 max|F| eV/A, |dE| <= 1e-4 + 1e-6 |E| eV)."""
import numpy as np
import pytest

from test_pbc import _set_pbc
from test_surface_atoms import molecule_over_slab

pytestmark = pytest.mark.gpu
SIZES = [4, 5, 7, 30, 63, 64, 65, 129]


def check(B, s, fo, Eo):
    d = np.abs(B.forces(s) - fo).max()
    assert d <= 1e-4 + 5e-6 * np.abs(fo).max(), (s, d, np.abs(fo).max())
    assert abs(B.E[s] - Eo) <= 1e-4 + 1e-6 * abs(Eo), (s, B.E[s], Eo)


@pytest.mark.parametrize("nPBC", [(0, 0, 0), (1, 0, 0), (4, 3, 0), (6, 2, 0), (2, 2, 1)])
def test_periodic(orc, nPBC):  # 1, 3, 63, 65 and 75 images
    from firecore_amd import native
    mols, cells = [], []
    for n in SIZES:
        m = native.gen_molecule(n, 40 + n, 0.05, n)
        p = m["apos"][:n]
        p -= p.mean(0)
        cells.append(np.diag(np.ptp(p, axis=0) + np.array([4.0, 5.0, 9.0])))
        if nPBC[0]:
            p[p[:, 0] > 0.5] += cells[-1][0]  # bonds to another image than the central one
        mols.append(m)
    native.init_systems(mols + [native.gen_molecule(33, 7, 0.05, 7)])
    for s, lvec in enumerate(cells):
        native.set_lattice(s, lvec, nPBC)
    print("case: non-bonded lanes, images", nPBC, flush=True)
    native.eval_forces()
    B = native.Batch()
    for s in range(B.nsys):
        m = B.system(s)
        if s < len(cells):
            _set_pbc(orc, m, cells[s], nPBC)
        try:
            fo, _, _, Eo = orc.eval(m)
        finally:
            orc.set_pbc()
        check(B, s, fo, Eo)


@pytest.mark.parametrize("nPBC", [(0, 0, 0), (2, 1, 0)])
def test_substrate_atoms(orc, nPBC):
    from firecore_amd import native
    native.init_systems([molecule_over_slab(n, 60 + n) for n in SIZES])
    native.attach_surface_atoms("synth:NaCl", nPBC)
    try:
        a, q, lv, _ = native.surface_atoms()
        orc.set_surface(a, q, lv, nPBC, 1.5)
        print("case: non-bonded lanes, substrate images", nPBC, flush=True)
        native.eval_forces()
        B = native.Batch()
        for s in range(B.nsys):
            fo, _, _, Eo = orc.eval(B.system(s))
            check(B, s, fo, Eo)
    finally:
        orc.set_surface()
        native.attach_surface_atoms(None)
