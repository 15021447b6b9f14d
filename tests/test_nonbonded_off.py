"""Relaxation with the non-bonded terms switched off: the pair loop is left out, and the
halves of a grid window, which stand before and in the middle of that loop, are still
sampled.  One wave and several, full and partly filled ones."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
SIZES = [4, 5, 24, 63, 64, 65, 129, 256]


@pytest.fixture
def no_pairs():
    from firecore_amd import MMFF_multi as mm
    mm.setSwitches_multi(NonBonded=-1)
    yield mm
    mm.setSwitches_multi(NonBonded=1)


@pytest.mark.parametrize("grid", [False, True])
def test_forces(orc, no_pairs, grid):
    """Exact forces after one move against the FP64 oracle (max|dF| <= 1e-4 + 5e-6 max|F|
    eV/A, the bound of the other force tests)."""
    from firecore_amd import native
    mols = [native.gen_molecule(n, 500 + n, 0.1, n) for n in SIZES]
    native.set_opt(0.1, 0.02, 0.2, 1.1, 0.5, 0.8, 5)
    native.set_force_limit(0.0)
    native.init_systems(mols)
    if grid:
        native.attach_surface("synth:NaCl", 0.1)
        top = native.grid_info()["pos0"][2]
        B = native.Batch()
        for s, n in enumerate(SIZES):
            p = B.atoms[B.info[s, 4]:B.info[s, 4] + n]
            p[:, 2] += top + 3.0 - p[:, 2].min()
        native.upload(False, False, False)
    print("case: no non-bonded terms, grid", grid, flush=True)
    native.relax(1, 1e-9, 0, False, True)
    B = native.Batch()
    g = native.grid_info() if grid else None
    for s, n in enumerate(SIZES):
        fo = orc.eval(dict(mols[s], apos=B.positions(s)), grid=g, sw=(1, 1, 1, 1, 0))[0]
        d = np.abs(B.forces(s) - fo).max()
        assert d <= 1e-4 + 5e-6 * np.abs(fo).max(), (n, d, np.abs(fo).max())


def test_no_time_for_pairs(no_pairs):
    """The pairs are about three quarters of a step of one molecule of 251 atoms."""
    from firecore_amd import native
    native.set_precond(0)
    native.set_force_limit(10.0)
    ms = {}
    for on in (-1, 1):
        no_pairs.setSwitches_multi(NonBonded=on)
        native.init_workload(1, 1, 10001, 251, 251, 0.1, None, 0.1)
        print("case: time without and with non-bonded terms", on, flush=True)
        for _ in range(5):
            native.relax(200, 1e-9, 0, True, False)
            ms[on] = min(ms.get(on, 1e9), native.last_ms())
    assert ms[-1] < 0.7 * ms[1], ms
