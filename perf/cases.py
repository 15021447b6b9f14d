"""The workloads whose speed this framework is measured by.

Every case goes through the public entry points (firecore_amd.native and
firecore_amd.MMFF_multi): new geometries are put into the host mirrors, uploaded,
worked on by the device and read back, as a program does that relaxes one set of
start geometries after another on a batch whose topology it keeps.

The headline relaxations run to convergence, each system to its own max|f|; the
others a fixed number of FIRE steps, the way frames are produced (MDloop's perframe;
the reference's own timings are for 100 steps).

Positions and energies are returned, forces where they are what was asked for.
Energies are handed out in double but are sums of FP32 terms, so they are returned
in FP32.

exact() is the same force field, FIRE and preconditioner in plain torch in 64 bits,
from the FP32 parameters that the device holds.
"""
import itertools
import math

import numpy as np
import torch

from firecore_amd import MMFF_multi, native

KQ = 14.3996448915  # eV*A/e^2
FIRE = (0.1, 0.02, 0.2, 1.1, 0.5, 0.8, 5)  # MMFF_multi.set_opt() defaults
FLIM = 10.0  # per-vec force clamp of the reference's update kernel, eV/A
SCAN_FLIM = 100.0  # scan()'s default
FCONV = 1e-3
GSTAR, GRIGID = 2.0, 127.0  # constant gains of the benchmark's ablation form
SURF_NPBC = (2, 2, 0)
CELL = 5.64  # A, period of the substrate


def _case(name, call, systems, nmin, nmax, mols="mixed", over="none", form="plain", steps=0, path="persistent"):
    """One case: `call` is what the program asks for, `mols` how the batch is made
    up (replicas of one molecule, mixed sizes, pairs of molecules, periodic
    molecules), `over` the substrate."""
    return dict(name=name, call=call, systems=systems, nmin=nmin, nmax=nmax, mols=mols, over=over, form=form,
                steps=steps, path=path)


def listed():
    return [
        # one small molecule, energy and forces: the smallest call, as a driver makes it that moves
        # the atoms itself (another optimiser, a finite-difference check)
        _case("forces_one_molecule", "forces", 1, 24, 24, "replicas"),
        # energy and forces of the headline batch: re-scoring of a whole screening set
        _case("forces_mixed_4096", "forces", 4096, 16, 256, "mixed", "grid"),
        # the shape of the reference's own published timings: 10 replicas, 100 FIRE steps
        _case("relax_10_replicas", "relax", 10, 24, 24, "replicas", steps=100),
        # 1024 replicas of one molecule in vacuum (conformers), to convergence
        _case("relax_1024_replicas", "relax", 1024, 24, 24, "replicas", steps=5000),
        # the headline batch, 16 to 256 atoms over the NaCl GridFF, in the reference's dynamics: the
        # part of a relaxation in which every system still moves
        _case("relax_mixed_4096_plain", "relax", 4096, 16, 256, "mixed", "grid", "plain", 1000),
        # the same with the trained proposal network and to convergence: the headline form
        _case("relax_mixed_4096_learned", "relax", 4096, 16, 256, "mixed", "grid", "learned", 10000),
        # the screening workload: pairs of molecules of 8 to 64 atoms each, at most 3000 steps
        _case("relax_pairs_8192_learned", "relax", 8192, 8, 64, "pairs", "grid", "learned", 3000),
        # one large molecule with an odd atom count: the latency of a step
        _case("relax_one_large", "relax", 1, 251, 251, "mixed", "grid", "constant", 200),
        # periodic molecules (a layer in its cell), which the split kernels relax
        _case("relax_periodic_32", "relax", 32, 40, 96, "periodic", "none", "plain", 30),
        # molecules over explicit substrate atoms instead of a grid
        _case("relax_over_atoms_64", "relax", 64, 16, 128, "mixed", "atoms", "plain", 30),
        # rigid placements of one molecule over the grid, relaxed with an anchored atom (scan)
        _case("scan_512_placements", "scan", 512, 36, 36, "replicas", "grid", "plain", 200),
        # one gradient of the proposal network's training: forward, loss and backward
        _case("network_gradient_512", "network", 512, 16, 256, "mixed", "grid", "learned"),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """A case of the listed ones' ranges."""
    what = rng.choice(["forces", "vacuum", "grid", "grid", "pairs", "large", "periodic", "atoms", "scan", "network"])
    form = rng.choice(["plain", "constant", "learned"])
    if what == "forces":
        nmax = _log(rng, 24, 256)
        return _draw("forces", _log(rng, 1, 4096), rng.randint(16, nmax), nmax, "mixed", rng.choice(["none", "grid"]))
    if what == "vacuum":
        n, path = _log(rng, 16, 128), rng.choice(["persistent", "persistent", "split"])
        return _draw("relax", _log(rng, 1, 2048), n, n, "replicas", form=rng.choice(["plain", "constant"]),
                     steps=rng.randint(10, 40) if path == "split" else _log(rng, 50, 2000), path=path)
    if what == "grid":
        nmax = _log(rng, 24, 256)
        return _draw("relax", _log(rng, 32, 4096), rng.randint(16, nmax), nmax, "mixed", "grid", form,
                     _log(rng, 100, 1000))
    if what == "pairs":
        nmax = _log(rng, 16, 64)
        return _draw("relax", _log(rng, 256, 8192), 8, nmax, "pairs", "grid", form, _log(rng, 100, 1000))
    if what == "large":
        n = rng.randint(129, 256)
        return _draw("relax", rng.randint(1, 16), n, n, "mixed", rng.choice(["none", "grid"]), form,
                     _log(rng, 100, 1000))
    if what == "periodic":
        nmax = rng.randint(32, 96)
        return _draw("relax", _log(rng, 1, 64), rng.randint(24, nmax), nmax, "periodic", steps=rng.randint(10, 30))
    if what == "atoms":
        nmax = rng.randint(24, 128)
        return _draw("relax", _log(rng, 1, 128), rng.randint(16, nmax), nmax, "mixed", "atoms",
                     steps=rng.randint(10, 30))
    if what == "scan":
        n = _log(rng, 16, 64)
        return _draw("scan", _log(rng, 8, 512), n, n, "replicas", "grid", steps=rng.randint(100, 200))
    nmax = _log(rng, 32, 256)
    return _draw("network", _log(rng, 16, 512), rng.randint(16, nmax), nmax, "mixed", "grid", "learned")


def _draw(*a, **k):
    c = _case("", *a, **k)
    del c["name"]
    return c


# ------------------------------------------------------------------ the batch
_loaded = {"key": None, "batch": None, "atoms": False}


def _key(case):
    return tuple(sorted((k, v) for k, v in case.items() if k != "name"))


def _periodic(case):
    """Molecules centred in one orthorhombic cell, with atoms moved across its
    faces so that bonds use other images than the central one."""
    mols = []
    for i in range(case["systems"]):
        n = case["nmin"] + (case["nmax"] - case["nmin"]) * i // max(case["systems"] - 1, 1)
        m = native.gen_molecule(n, 30001 + i, 0.05, 30001 + i)
        m["apos"][:n] -= m["apos"][:n].mean(0)
        mols.append(m)
    size = np.max([np.ptp(m["apos"][:m["natoms"]], axis=0) for m in mols], axis=0)
    lvec = np.diag(size + np.array([3.0, 3.0, 12.0]))
    for m in mols:
        p = m["apos"][:m["natoms"]]
        p[p[:, 0] > 0.5] -= lvec[0]
        p[(p[:, 1] > 0.8) & (np.arange(len(p)) % 2 == 0)] -= lvec[1]
    return mols, lvec


def _load(case):
    """The case's batch in the library, and the settings a program gives it."""
    if _loaded["key"] == _key(case):
        return _loaded["batch"]
    _loaded["key"] = None
    ns, nmin, nmax = case["systems"], case["nmin"], case["nmax"]
    surf = "synth:NaCl" if case["over"] == "grid" else None
    native.set_precond(0)
    if _loaded["atoms"]:
        native.attach_surface_atoms(None)
    _loaded["atoms"] = case["over"] == "atoms"
    native.set_opt(*FIRE)
    native.set_force_limit(FLIM)
    if case["call"] == "scan":
        MMFF_multi.init(nSys_=1, xyz_name="synth:natoms=%d,seed=0,sigma=0" % nmin, surf_name=surf, nPBC=(0, 0, 0))
    elif case["mols"] == "periodic":
        mols, lvec = _periodic(case)
        native.init_systems(mols)
        native.set_lattice(-1, lvec, (1, 1, 0))
    else:
        kind = {"replicas": 0, "mixed": 1, "pairs": 2}[case["mols"]]
        native.init_workload(kind, ns, {0: 0, 1: 10001, 2: 20001}[kind], nmin, nmax, 0.1, surf, 0.1)
    B = native.Batch()
    if case["over"] == "atoms":
        # neutral molecules lowered onto the slab: under the bare Coulomb of explicit ions a
        # randomly charged atom falls onto an ion
        native.attach_surface_atoms("synth:NaCl", SURF_NPBC)
        top = native.surface_atoms()[0][:, 2].max()
        B.REQs[:, 2] = 0.0
        for s in range(B.nsys):
            n, v0 = int(B.info[s, 0]), int(B.info[s, 4])
            p = B.atoms[v0:v0 + n]
            p[:, :3] -= p[:, :3].mean(0)
            p[:, 2] += top + 3.0 - p[:, 2].min()
        native.upload(True, False, False)
    if case["form"] == "learned":
        native.set_proposal_weights(np.load("firecore_amd/proposal_weights.npy"))
        native.set_proposal_every(128)
        native.set_precond(2, 3.0, 127.0)
    elif case["form"] == "constant":
        native.set_precond(1, GSTAR, GRIGID)
    _loaded.update(key=_key(case), batch=B, base=B.atoms.copy())
    return B


def prepare(case, seed):
    """Start geometries: each molecule of the batch moved over the substrate and
    its atoms displaced; for scan(), placements of its template."""
    B = _load(case)
    rng = np.random.default_rng(seed)
    if case["call"] == "scan":
        n = case["systems"]
        q = rng.normal(size=(n, 4))
        a, b, c, d = (q / np.linalg.norm(q, axis=1, keepdims=True)).T
        rots = np.stack([a * a + b * b - c * c - d * d, 2 * (b * c - a * d), 2 * (b * d + a * c),
                         2 * (b * c + a * d), a * a - b * b + c * c - d * d, 2 * (c * d - a * b),
                         2 * (b * d - a * c), 2 * (c * d + a * b), a * a - b * b - c * c + d * d], 1).reshape(n, 3, 3)
        tmpl = native.gen_molecule(case["nmin"], 0)["apos"]
        z = np.einsum("ia,naq->niq", tmpl[:case["nmin"]], rots)[:, :, 2].min(1)
        top = native.grid_info()["pos0"][2]
        poss = np.concatenate([rng.uniform(0, CELL, (n, 2)), (top + 3.0 - z)[:, None]], 1)
        return dict(case=case, poss=np.ascontiguousarray(poss), rots=np.ascontiguousarray(rots))
    atoms = _loaded["base"].copy()
    info = B.info
    N, v0 = info[:, 0].astype(np.int64), info[:, 4].astype(np.int64)
    rows = np.repeat(v0, N) + np.arange(N.sum()) - np.repeat(np.cumsum(N) - N, N)
    shift = np.zeros((len(N), 3))
    if case["over"] != "none":
        shift[:, :2] = rng.uniform(0, CELL, (len(N), 2))
    atoms[rows, :3] += (np.repeat(shift, N, axis=0) + rng.normal(0.0, 0.02, (len(rows), 3))).astype(np.float32)
    return dict(case=case, atoms=atoms)


def run(state):
    case = state["case"]
    B = _load(case)
    if case["call"] == "scan":
        n, na = case["systems"], case["nmin"]
        E, pos = np.zeros(n), np.zeros((n, na, 3))
        MMFF_multi.scan(state["poss"], state["rots"], Es=E, aposs=pos, bRelax=True, niter_max=case["steps"],
                        Fconv=FCONV, Flim=SCAN_FLIM)
        return {"energy": E.astype(np.float32), "positions": pos.astype(np.float32)}
    B.atoms[:] = state["atoms"]
    native.upload(False, False, False)
    if case["call"] == "forces":
        native.eval_forces()
        return {"energy": B.E.astype(np.float32), "forces": B.aforces[:, :3].copy()}
    if case["call"] == "network":
        out, _ = native.proposal_forward()
        dout, loss = native.proposal_loss_grad(0.02, 0.5)
        return {"outputs": out, "loss": loss, "gradient": native.proposal_backward(dout)}
    native.relax(case["steps"], FCONV, 1 if case["path"] == "split" else 0, False, True)
    return {"energy": B.E.astype(np.float32), "positions": B.atoms[:, :3].copy()}


def work(case):
    """Pairs 38 FLOP, grid sample 740 and 64 coefficients per atom, bonded terms
    400 per node, FIRE 40 per vec, explicit substrate atom 30 per image; the
    bytes are the batch once in and the results once out."""
    ns, lo, hi = case["systems"], case["nmin"], case["nmax"]
    sizes = np.arange(lo, hi + 1.0)
    n, n2 = sizes.mean(), (sizes ** 2).mean()
    if case["mols"] == "pairs":
        n, n2 = 2 * n, 2 * n2 + 2 * n * n
    images = 9 if case["mols"] == "periodic" else 1
    step = 38 * n2 / 2 * images + 400 * 0.45 * n + 40 * 1.45 * n
    step += {"none": 0, "grid": 740, "atoms": 30 * 8 * 25}[case["over"]] * n
    evals = min(case["steps"], 1800) + 1  # about where the mean system converges
    flops = step * evals
    if case["call"] == "network":
        flops = 2 * step + 3 * 35.1e3 * n
    elif case["form"] == "learned":
        flops += 35.1e3 * n * (1 + case["steps"] // 128) + 150 * n * evals
    byts = n * (1.45 * 16 * 3 + 16 * 4 + 0.45 * 80 + n / 8)
    return {"bytes": float(ns * byts), "flops": float(ns * flops)}


# ------------------------------------------------------------- 64-bit values
def exact(case, seed):
    if case["form"] == "learned":
        return None  # its gains come from BF16 products, which have no value in 64 bits
    if case["steps"] > 200:
        return None  # by then rounding alone decides where some of the systems go
    state = prepare(case, seed)
    F = _ForceField(case, state)
    if F.pairs * (case["steps"] + 1) > 1e10:
        return None  # would take minutes
    steps = case["steps"]
    out = [g.relax(steps, SCAN_FLIM if case["call"] == "scan" else FLIM) if steps else g.forces() for g in F.groups]
    energy = np.zeros(F.nsys)
    vecs = np.zeros((F.nvec, 3))
    for g, (E, p, h) in zip(F.groups, out):
        energy[g.ids] = E.cpu().numpy()
        p, h = p.cpu().numpy(), h.cpu().numpy()
        for k in range(len(g.ids)):
            n, m, v0 = g.n[k], g.m[k], g.v0[k]
            vecs[v0:v0 + n], vecs[v0 + n:v0 + n + m] = p[k, :n], h[k, :m]
    if case["call"] == "scan":
        vecs = vecs.reshape(F.nsys, -1, 3)[:, :case["nmin"]]
    return {"energy": energy, "forces" if case["call"] == "forces" else "positions": vecs}


def _components(n, neighs, most=4):
    label = np.arange(n)
    i, k = np.nonzero(neighs >= 0)
    j = neighs[i, k]
    while True:
        new = label.copy()
        np.minimum.at(new, i, label[j])
        np.minimum.at(new, j, label[i])
        if (new == label).all():
            return np.minimum(np.unique(label, return_inverse=True)[1], most - 1)
        label = new


class _ForceField:
    """The batch of a case in groups of similar size, padded."""

    def __init__(self, case, state):
        B = _load(case)
        d = {k: np.array(getattr(B, k)) for k in
             ("REQs", "PLQs", "neighs", "MMpars", "BLs", "BKs", "Ksp", "Kpp")}
        info = np.array(B.info[:, :5]).astype(np.int64)
        anchor = None
        if case["call"] == "scan":  # every placement has the template's parameters
            n, m = case["nmin"], int(info[0, 1])
            a = np.einsum("va,naq->nvq", native.gen_molecule(n, 0)["apos"], state["rots"])
            a[:, :n] += state["poss"][:, None]
            atoms = a.astype(np.float32).astype(np.float64).reshape(-1, 3)
            ns = case["systems"]
            s = np.arange(ns)
            info = np.stack([np.full(ns, n), np.full(ns, m), 0 * s, 0 * s, s * (n + m)], 1)
            anchor = torch.tensor(state["poss"].astype(np.float32).astype(np.float64))
        else:
            atoms = state["atoms"][:, :3].astype(np.float64)
        self.nsys, self.nvec = len(info), len(atoms)
        shifts, cells = np.zeros((1, 3)), None
        if case["mols"] == "periodic":
            base = _loaded["base"].astype(np.float64)
            lvec = _periodic(case)[1]
            shifts = np.array([x * lvec[0] + y * lvec[1] for y in (-1, 0, 1) for x in (-1, 0, 1)])
            cells = np.full(d["neighs"].shape, -1)
            for n, m, a0, n0, v0 in info:  # the image of each bond: the nearest one
                nb = d["neighs"][a0:a0 + n]
                p = base[v0:v0 + n, :3]
                r = p[np.maximum(nb, 0)][:, :, None] + shifts[None, None] - p[:, None, None]
                cells[a0:a0 + n] = np.where(nb >= 0, (r ** 2).sum(-1).argmin(-1), -1)
            shifts = shifts.astype(np.float32).astype(np.float64)
        self.pairs = float((info[:, 0] ** 2).sum()) * len(shifts)
        order = np.argsort(info[:, 0], kind="stable")
        self.groups, at = [], 0
        while at < len(order):
            upto = at + 1
            while upto < len(order) and (upto + 1 - at) * info[order[upto], 0] ** 2 < 4e6:
                upto += 1
            self.groups.append(_Group(case, order[at:upto], info, d, atoms, shifts, cells, anchor))
            at = upto


class _Group:
    def __init__(self, case, ids, info, d, atoms, shifts, cells, anchor):
        self.case, self.ids = case, ids
        self.n, self.m, self.v0 = info[ids, 0], info[ids, 1], info[ids, 4]
        dev = "cuda" if torch.cuda.is_available() else "cpu"
        T = lambda x: torch.as_tensor(np.ascontiguousarray(x), device=dev)
        S, N, M = len(ids), int(self.n.max()), int(self.m.max())

        def pad(src, rows, most, off, fill=0.0):
            out = np.full((S, most) + src.shape[1:], fill, src.dtype if src.dtype.kind == "i" else np.float64)
            for k in range(S):
                out[k, :rows[k]] = src[off[k]:off[k] + rows[k]]
            return out
        a0, n0 = info[ids, 2], info[ids, 3]
        self.p, self.h = T(pad(atoms, self.n, N, self.v0)), T(pad(atoms, self.m, M, self.v0 + self.n))
        self.atom = T(np.arange(N)[None] < self.n[:, None])
        self.node = T(np.arange(M)[None] < self.m[:, None])
        self.REQ = T(pad(d["REQs"], self.n, N, a0))
        self.PLQ = T(pad(d["PLQs"], self.n, N, a0))
        nb = pad(d["neighs"], self.n, N, a0, -1).astype(np.int64)
        self.nb = T(nb[:, :M])
        self.has = (self.nb >= 0) & self.node[..., None]
        self.apar, self.bL, self.bK, self.ksp, self.kpp = (
            T(pad(d[k], self.m, M, n0)) for k in ("MMpars", "BLs", "BKs", "Ksp", "Kpp"))
        self.shifts = T(shifts)
        nc = pad(cells, self.n, N, a0, -1).astype(np.int64) if cells is not None else np.where(nb >= 0, 0, -1)
        self.bshift = self.shifts[T(np.maximum(nc[:, :M], 0))] * (1.0 if cells is not None else 0.0)
        # pairs of the non-bonded sum: all but an atom with itself and with its neighbours (at the bond's image)
        w = (self.atom[:, None, :, None] & self.atom[:, None, None, :]).double().repeat(1, len(shifts), 1, 1)
        w[:, :, range(N), range(N)] = 0.0
        s, i, k = np.nonzero(nb >= 0)
        w[T(s), T(nc[s, i, k]), T(i), T(nb[s, i, k])] = 0.0
        self.w = w
        if case["form"] == "constant":
            comp = np.zeros((S, N), np.int64)
            for k in range(S):
                comp[k, :self.n[k]] = _components(int(self.n[k]), nb[k, :self.n[k]])
            self.comp = T(comp)
        if case["over"] == "grid":
            g = native.grid_info()
            self.gn, self.g0 = g["n"], T(g["pos0"].astype(np.float32).astype(np.float64))
            self.gi = T((1.0 / g["step"]).astype(np.float32).astype(np.float64))
            self.gc = T(np.asarray(g["coefs"]).reshape(-1, 3).astype(np.float32)).double()
        elif case["over"] == "atoms":
            sp, sq, lv, _ = native.surface_atoms()
            img = np.array([x * lv[0] + y * lv[1] for x, y in itertools.product(range(-2, 3), range(-2, 3))])
            f32 = lambda x: x.astype(np.float32).astype(np.float64)
            self.sp = T((f32(sp)[:, None] + f32(img)[None]).reshape(-1, 3))
            self.sq = T(np.repeat(f32(sq), len(img), axis=0))
        self.anchor = None if anchor is None else anchor[torch.as_tensor(ids)].to(dev)

    def gather(self, x):
        """x of every node's four neighbours."""
        S, M = self.nb.shape[:2]
        return torch.gather(x, 1, self.nb.clamp(min=0).reshape(S, M * 4, 1).expand(-1, -1, 3)).reshape(S, M, 4, 3)

    def scatter(self, out, x):
        S, M = self.nb.shape[:2]
        x = torch.where(self.has[..., None], x, torch.zeros_like(x))
        out.scatter_add_(1, self.nb.clamp(min=0).reshape(S, M * 4, 1).expand(-1, -1, 3), x.reshape(S, M * 4, 3))

    @staticmethod
    def pair(d, a, b):
        """Force factor and energy of the pair of parameters a and b at d."""
        r2 = (d * d).sum(-1)
        ir2 = 1.0 / r2
        e0, q = a[..., 1] * b[..., 1], KQ * a[..., 2] * b[..., 2] * ir2.sqrt()
        u6 = ((a[..., 0] + b[..., 0]) ** 2 * ir2) ** 3
        hb = u6 * u6 * (a[..., 3] * b[..., 3]).clamp(max=0.0) * e0
        v = u6 * e0
        return (q + 12.0 * ((u6 - 1.0) * v + hb)) * ir2, q + (u6 - 2.0) * v + hb

    def forces(self, p=None, h=None):
        """Energy, forces on the atoms and on the pi-vectors."""
        p, h = (self.p if p is None else p), (self.h if h is None else h)
        S, N = p.shape[:2]
        f, fh = torch.zeros_like(p), torch.zeros_like(h)
        E = torch.zeros(S, dtype=p.dtype, device=p.device)
        for k in range(len(self.shifts)):  # non-bonded pairs
            d = p[:, None] - p[:, :, None] + self.shifts[k]
            w = self.w[:, k]
            d = torch.where(w[..., None] != 0, d, torch.ones_like(d))
            fr, e = self.pair(d, self.REQ[:, :, None], self.REQ[:, None])
            f -= (d * (fr * w)[..., None]).sum(2)
            E += 0.5 * (e * w).sum((1, 2))
        # bonded terms of every node
        zero = torch.zeros((), dtype=p.dtype, device=p.device)
        M = h.shape[1]
        d = torch.where(self.has[..., None], self.gather(p) + self.bshift - p[:, :M, None], torch.ones_like(p[:, :M, None]))
        l = d.norm(dim=-1)
        u = d / l[..., None]
        rec, recpi = torch.zeros_like(d), torch.zeros_like(d)
        own = torch.arange(M, device=p.device)[None, :, None]
        first = self.has & (own < self.nb)
        dl = torch.where(first, l - self.bL, zero)
        E += 0.5 * (self.bK * dl * dl).sum((1, 2))
        fb = u * (self.bK * dl)[..., None]
        rec -= fb
        fa = fb.sum(2)
        pp = first & (self.nb < torch.as_tensor(self.m, device=p.device)[:, None, None]) & (self.kpp > 1e-6)
        hp = torch.gather(h, 1, self.nb.clamp(0, M - 1).reshape(S, M * 4, 1).expand(-1, -1, 3)).reshape(S, M, 4, 3)
        c = (h[:, :, None] * hp).sum(-1)
        K = torch.where(pp, self.kpp, zero)
        E += (K * (1.0 - c.abs())).sum((1, 2))
        K = torch.where(c < 0, -K, K)[..., None]
        fh += ((hp - h[:, :, None] * c[..., None]) * K).sum(2)
        recpi += (h[:, :, None] - hp * c[..., None]) * K
        ps = self.has & (self.ksp > 1e-6)
        c = (h[:, :, None] * u).sum(-1)
        c_ = torch.where(ps, c - self.apar[..., 3:], zero)
        K = torch.where(ps, self.ksp, zero)
        E += (K * c_ * c_).sum((1, 2))
        fang = (-2.0 * K * c_)[..., None]
        fh += ((u - h[:, :, None] * c[..., None]) * fang).sum(2)
        f2 = (h[:, :, None] - u * c[..., None]) * fang / l[..., None]
        fa -= f2.sum(2)
        rec += f2
        nREQ = torch.stack([torch.gather(self.REQ, 1, self.nb[..., k].clamp(min=0)[..., None].expand(-1, -1, 4))
                            for k in range(4)], 2)
        for a, b in itertools.combinations(range(4), 2):  # angles, and the 1-3 pair taken out of the sum above
            ok = (self.has[:, :, a] & self.has[:, :, b])[..., None]
            s = u[:, :, a] + u[:, :, b]
            c2 = (s * s).sum(-1) * 0.25
            c2 = torch.where(ok[..., 0], c2, 0.5 + 0 * c2)
            c, sn = c2.sqrt(), (1.0 - c2).clamp(min=1e-14).sqrt()
            x, y = self.apar[..., 0] * c + self.apar[..., 1] * sn, self.apar[..., 1] * c - self.apar[..., 0] * sn
            K = torch.where(ok[..., 0], self.apar[..., 2], zero)
            E += (K * y * y / (1.0 + x)).sum(1)
            g = (-K * y / (4.0 * c * sn))[..., None]
            both = torch.zeros_like(fa)
            for q in (a, b):
                t = (s - 2.0 * c2[..., None] * u[:, :, q]) * g / l[:, :, q, None]
                rec[:, :, q] += t
                both += t
            fa -= both
            dd = torch.where(ok, d[:, :, b] - d[:, :, a], torch.ones_like(fa))
            fr, e = self.pair(dd, nREQ[:, :, a], nREQ[:, :, b])
            t = torch.where(ok, dd * fr[..., None], torch.zeros_like(dd))
            rec[:, :, a] += t
            rec[:, :, b] -= t
            E -= torch.where(ok[..., 0], e, zero).sum(1)
        f[:, :M] += fa
        self.scatter(f, rec)
        t = torch.zeros_like(f)
        self.scatter(t, recpi)
        fh = fh + t[:, :M]
        if self.case["over"] == "grid":
            e, fg = self.grid(p.reshape(-1, 3), self.PLQ.reshape(-1, 4)[:, :3])
            E += (e.reshape(S, N) * self.atom).sum(1)
            f += fg.reshape(S, N, 3)
        elif self.case["over"] == "atoms":
            d = torch.where(self.atom[..., None, None], p[:, :, None] - self.sp, torch.ones_like(p[:, :1, None]))
            r2 = (d * d).sum(-1)
            r = r2.sqrt()
            e = torch.exp(-1.5 * (r - self.sq[:, 0] - self.REQ[..., 0, None]))
            A = e * self.sq[:, 1] * self.REQ[..., 1, None]
            q = KQ * self.sq[:, 2] * self.REQ[..., 2, None] / r
            E += ((A * (e - 2.0) + q).sum(2) * self.atom).sum(1)
            f -= (d * (-3.0 * A * (e - 1.0) / r - q / r2)[..., None]).sum(2)
        if self.anchor is not None:
            f[:, 0] += self.anchor - p[:, 0]
        fh = fh - h * (h * fh).sum(-1, keepdim=True)
        return E, f * self.atom[..., None], fh * self.node[..., None]

    def grid(self, p, plq):
        """Tricubic B-spline sample of the substrate's three channels."""
        u = (p - self.g0) * self.gi
        i = torch.cat([u[:, :2].floor(), u[:, 2:].trunc()], 1)
        t = u - i
        i = i.long()
        nx, ny, nz = self.gn
        iz = i[:, 2].clamp(3, nz - 5)
        b = torch.stack([(1 - t) ** 3 / 6, (3 * t ** 3 - 6 * t ** 2 + 4) / 6,
                         (3 * t + 3 * t ** 2 - 3 * t ** 3 + 1) / 6, t ** 3 / 6], -1)
        db = torch.stack([-0.5 * (1 - t) ** 2, 0.5 * (3 * t ** 2 - 4 * t), 0.5 * (-3 * t ** 2 + 2 * t + 1),
                          0.5 * t ** 2], -1)
        o = torch.arange(4, device=p.device) - 1
        X, Y, Z = (i[:, :1] + o) % nx, (i[:, 1:2] + o) % ny, iz[:, None] + o
        E, f = torch.zeros_like(p[:, 0]), torch.zeros_like(p)
        for lo in range(0, len(p), 100000):
            q = slice(lo, lo + 100000)
            at = ((X[q, :, None] * ny + Y[q, None])[..., None] * nz + Z[q, None, None])
            c = (self.gc[at] * plq[q, None, None, None]).sum(-1)
            k = lambda x, y, z: torch.einsum("nabc,na,nb,nc->n", c, x[q, 0], y[q, 1], z[q, 2])
            E[q] = k(b, b, b)
            f[q] = -torch.stack([k(db, b, b), k(b, db, b), k(b, b, db)], -1) * self.gi
        return E, f

    def precondition(self, p, f):
        """Rigid-body projections of the force on stars and components, added with their gains."""
        def turn(r, fr, ok):  # mean force and angular rate of groups (..., members, 3)
            n = ok.sum(-1, keepdim=True)
            w = ok[..., None]
            c = (r * w).sum(-2) / n.clamp(min=1)
            t = (fr * w).sum(-2) / n.clamp(min=1)
            q = (r - c[..., None, :]) * w
            L = torch.cross(q, fr * w, dim=-1).sum(-2)
            q2 = (q * q).sum((-1, -2))[..., None, None]
            eye = torch.eye(3, dtype=p.dtype, device=p.device)
            I = q2 * eye - q.transpose(-1, -2) @ q
            tr = I.diagonal(dim1=-2, dim2=-1).sum(-1)[..., None, None]
            I = I + (1e-6 * tr + 1e-20) * eye
            I = torch.where(n[..., None] < 3, q2.clamp(min=1e-20) * eye, I)
            return c, t, torch.linalg.solve(I, L[..., None])[..., 0]
        S, N = p.shape[:2]
        M = self.nb.shape[1]
        ok = torch.cat([self.node[..., None], self.has], -1).double()
        r = torch.cat([p[:, :M, None], self.gather(p)], 2)
        fr = torch.cat([f[:, :M, None], self.gather(f)], 2)
        c, t, w = turn(r, fr, ok)
        d = (t[:, :, None] + torch.cross(w[:, :, None].expand_as(r), r - c[:, :, None], dim=-1)) * GSTAR * ok[..., None]
        out = f.clone()
        out[:, :M] += d[:, :, 0]
        self.scatter(out, d[:, :, 1:])
        for k in range(int(self.comp.max()) + 1):
            ok = (self.atom & (self.comp == k)).double()
            c, t, w = turn(p, f, ok)
            out += (t[:, None] + torch.cross(w[:, None].expand_as(p), p - c[:, None], dim=-1)) * GRIGID * ok[..., None]
        return out

    def relax(self, steps, flim):
        """FIRE with one state per system; energy and positions after `steps` moves."""
        p, h = self.p.clone(), self.h.clone()
        vp, vh = torch.zeros_like(p), torch.zeros_like(h)
        dt_max, dt_min, damp_max, finc, fdec, falpha, nlast = FIRE
        dt = torch.full((len(p),), dt_max, dtype=p.dtype, device=p.device)
        damp, last = torch.full_like(dt, damp_max), torch.zeros_like(dt)
        on = torch.ones_like(dt, dtype=torch.bool)
        for step in range(steps + 1):
            E, f, fh = self.forces(p, h)
            top = torch.maximum((f * f).sum(-1).amax(1), (fh * fh).sum(-1).amax(1))
            on = on & (top >= FCONV ** 2)
            if step == steps or not bool(on.any()):
                return E, p, h
            if self.case["form"] == "constant":
                f = self.precondition(p, f)
            clamp = lambda x: x * (flim / x.norm(dim=-1, keepdim=True).clamp(min=flim))
            f, fh = clamp(f), clamp(fh)
            dot = lambda a, b, c, d: (a * b).sum((1, 2)) + (c * d).sum((1, 2))
            vf, vv, ff = dot(vp, f, vh, fh), dot(vp, vp, vh, vh), dot(f, f, fh, fh)
            back = vf < 0
            renorm = (vv / ff.clamp(min=1e-60)).sqrt()
            cv = torch.where(back, 0 * dt, 1.0 - damp)
            cf = torch.where(back, 0 * dt, damp) * renorm * renorm
            grow = ~back & (last > nlast)
            dt = torch.where(back, (dt * fdec).clamp(min=dt_min), torch.where(grow, (dt * finc).clamp(max=dt_max), dt))
            damp = torch.where(back, 0 * damp + damp_max, torch.where(grow, damp * falpha, damp))
            last = torch.where(back, 0 * last, last + 1)
            B = lambda x: x[:, None, None]
            fh = fh - h * (h * fh).sum(-1, keepdim=True)
            vp2, vh2 = vp * B(cv) + f * B(dt + cf), vh * B(cv) + fh * B(dt + cf)
            vh2 = vh2 - h * (h * vh2).sum(-1, keepdim=True)
            h2 = h + vh2 * B(dt)
            h2 = h2 / h2.norm(dim=-1, keepdim=True).clamp(min=1e-30)
            m = B(on)
            p, h = torch.where(m, p + vp2 * B(dt), p), torch.where(m, h2, h)
            vp, vh = torch.where(m, vp2, vp), torch.where(m, vh2, vh)
