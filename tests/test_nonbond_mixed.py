"""Non-bonded forces of large batches that hold both periodic and vacuum molecules, or
substrate atoms: the vacuum molecules go to a thread per atom, the periodic ones to a wave
per atom in the same launch, wherever in the batch they are.  Small batches take a wave
per atom for all.  Device forces and energies against the FP64 oracle (max|dF| <= 1e-4 +
5e-6 max|F| eV/A, |dE| <= 1e-4 + 1e-6 |E| eV)."""
import numpy as np
import pytest

from test_nonbond_lanes import check
from test_pbc import _set_pbc
from test_surface_atoms import molecule_over_slab

pytestmark = pytest.mark.gpu
SIZES = [4, 30, 63, 64, 65, 129]
NPBC = (1, 1, 0)


def periodic(n):
    from firecore_amd import native
    m = native.gen_molecule(n, 40 + n, 0.05, n)
    p = m["apos"][:n]
    p -= p.mean(0)
    cell = np.diag(np.ptp(p, axis=0) + np.array([4.0, 5.0, 9.0]))
    p[p[:, 0] > 0.5] += cell[0]
    return m, cell


def batch(copies, where):
    """Vacuum molecules of SIZES, `copies` times, with periodic ones put in before
    positions `where`; (molecule, cell or None) of each system."""
    from firecore_amd import native
    vac = [native.gen_molecule(n, 80 + n, 0.05, n) for n in SIZES] * copies
    out, sizes = [], iter(SIZES * len(where))
    for k in range(len(vac) + 1):
        if k in where:
            out.append(periodic(next(sizes)))
        if k < len(vac):
            out.append((vac[k], None))
    native.init_systems([m for m, _ in out])
    for s, (_, cell) in enumerate(out):
        if cell is not None:
            native.set_lattice(s, cell, NPBC)
    return out


def compare(orc, out, systems, g=None, energy=True):
    from firecore_amd import native
    B = native.Batch()
    for s in systems:
        m = B.system(s)
        if out[s][1] is not None:
            _set_pbc(orc, m, out[s][1], NPBC)
        try:
            fo, _, _, Eo = orc.eval(m, grid=g)
        finally:
            orc.set_pbc()
        check(B, s, fo, Eo if energy else B.E[s])


@pytest.mark.parametrize("copies", [1, 80])
@pytest.mark.parametrize("grid", [False, True])
def test_periodic_among_vacuum(orc, copies, grid):
    from firecore_amd import native
    last = copies * len(SIZES)
    where = {0, 2, last // 2, last}
    out = batch(copies, where)
    if grid:
        native.attach_surface("synth:NaCl", 0.1)
        B = native.Batch()
        for s in range(B.nsys):
            p = B.atoms[B.info[s, 4]:B.info[s, 4] + B.info[s, 0]]
            p[:, 2] += native.grid_info()["pos0"][2] + 3.0 - p[:, 2].min()
        native.upload(False, False, False)
    print("case: periodic among vacuum", copies, grid, flush=True)
    native.eval_forces()
    some = sorted({s for s, (_, c) in enumerate(out) if c is not None} | set(range(6)) | {len(out) - 2, len(out) // 2 + 1})
    compare(orc, out, some, native.grid_info() if grid else None)


def test_one_periodic_molecule_leaves_the_others_their_kernel():
    """A wave for every atom of 512 molecules of 256 takes three times as long over the grid
    as a thread."""
    from firecore_amd import native
    native.set_precond(0)
    big = native.gen_molecule(256, 336, 0.05, 256)
    ms = {}
    for extra in ([], [periodic(30)]):
        native.init_systems([big] * 512 + [m for m, _ in extra])
        native.attach_surface("synth:NaCl", 0.1)
        for _, cell in extra:
            native.set_lattice(512, cell, NPBC)
        print("case: time of 512 vacuum molecules and periodic ones:", len(extra), flush=True)
        for _ in range(5):
            native.relax(10, 1e-9, 1, True, False)
            ms[len(extra)] = min(ms.get(len(extra), 1e9), native.last_ms())
    assert ms[1] < 1.5 * ms[0], ms


@pytest.mark.parametrize("nPBC", [(0, 0, 0), (2, 1, 0)])
def test_many_over_substrate_atoms(orc, nPBC):
    from firecore_amd import native
    native.init_systems([molecule_over_slab(n, 60 + n) for n in SIZES] * 120)
    native.attach_surface_atoms("synth:NaCl", nPBC)
    try:
        a, q, lv, _ = native.surface_atoms()
        orc.set_surface(a, q, lv, nPBC, 1.5)
        print("case: many over substrate atoms", nPBC, flush=True)
        native.eval_forces()
        B = native.Batch()
        for s in list(range(7)) + [B.nsys - 1]:
            fo, _, _, Eo = orc.eval(B.system(s))
            check(B, s, fo, Eo)
    finally:
        orc.set_surface()
        native.attach_surface_atoms(None)


def test_split_part_of_a_relaxation(orc):
    """Periodic molecules and one of more than 256 atoms are relaxed after the others:
    exact forces at the geometries that come back."""
    from firecore_amd import native
    out = [(native.gen_molecule(40, 7, 0.05, 7), None), periodic(30), (native.gen_molecule(300, 8, 0.05, 8), None),
           periodic(65), (native.gen_molecule(64, 9, 0.05, 9), None)]
    native.set_precond(0)
    native.set_force_limit(0.0)
    native.set_opt(0.02, 0.005, 0.2, 1.1, 0.5, 0.8, 5)
    native.init_systems([m for m, _ in out])
    for s, (_, cell) in enumerate(out):
        if cell is not None:
            native.set_lattice(s, cell, NPBC)
    print("case: split part of a relaxation", flush=True)
    native.relax(2, 1e-9, 0, False, True)
    assert (np.array(native.Batch().nsteps) == 2).all()
    # the energy of 300 atoms differs by the rounding of their angle parameters alone
    compare(orc, out, range(len(out)), energy=False)
