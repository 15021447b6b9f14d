"""The persistent kernel's wave-wide refill of the GridFF window slots.

A relaxation of a few steps moves atoms across cell faces of the grid, so the
final forces are sampled through slots that were filled in different steps, by
waves that are full, hold one atom, or end inside the batch's last slots.  The
exact forces at the final geometry are compared with the FP64 oracle there
(max|dF| <= 1e-4 + 5e-6 max|F| eV/A, the bound of the other force tests; the
energy pass does not go through the slots).  Molecules lie at both sides of the cell's faces and up
to several cells away, below the grid's first nodes and above its last.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("natoms", [4, 63, 64, 65, 129, 256])
def test_forces_after_cell_crossings(orc, natoms):
    from firecore_amd import native
    print("case: grid window", natoms, flush=True)
    native.set_opt(0.1, 0.02, 0.2, 1.1, 0.5, 0.8, 5)
    native.set_force_limit(0.0)
    native.init_workload(1, 6, 50001, natoms, natoms, 0.02, "synth:NaCl", 0.1)
    B = native.Batch()
    g = native.grid_info()
    size = np.array(g["n"]) * g["step"]
    shift = [(0, 0, 0), (-0.5 * size[0], 0, 0), (size[0] * 2.5, -size[1] * 3.5, 0), (0.05, -0.05, 0),
             (0, 0, size[2]), (-size[0], size[1], -2.0)]
    for s in range(B.nsys):
        v0 = int(B.info[s, 4])
        B.atoms[v0:v0 + natoms, :3] += np.array(shift[s], np.float32)
    native.upload(False, False, False)
    native.relax(12, 1e-6, 0, False, True)
    # far above the grid the z-clamp extrapolates the spline, and unclamped forces may
    # throw a molecule out; the others have to take every step
    ok = [s for s in range(B.nsys) if not (s == 4 and B.status[s] == native.ST_NAN)]
    assert (np.array(B.nsteps)[ok] == 12).all()
    moved = 0
    for s in ok:
        m = B.system(s)
        fo = orc.eval(m, grid=g)[0]
        d = np.abs(B.forces(s) - fo).max()
        assert d <= 1e-4 + 5e-6 * np.abs(fo).max(), (s, d, np.abs(fo).max())
        m0 = native.gen_workload_system(1, s, 50001, natoms, natoms, 0.02, g)
        p0 = m0["apos"][:natoms] + np.array(shift[s])
        moved += int((np.floor(p0 / g["step"]) != np.floor(m["apos"][:natoms] / g["step"])).any(1).sum())
    assert moved > 0  # atoms did cross cell faces
