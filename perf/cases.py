"""The work that users of this library have it do, case by case, through its
public entry points: whole homogenizations of new images (compute_property and
the model entry points behind the command line), the batched solver, and
inference and training of the learned initial guess.

Sizes come from the repository's own workloads (32^3 conduction, 100^3 images,
128^3 and 256^3 elastic spheres, porous spheres, batches of uneven samples,
64^3 training images); others are generic and odd.  A homogenization is always
the whole call on an image the process has not seen: reading the model, maps,
upload, solver set-up, solve, effective matrix, release.

exact() solves the same discrete problems in plain torch FP64: conduction and
elasticity by CG preconditioned with the homogeneous medium in Fourier space,
Stokes flow by MINRES, the network with autograd.
"""
import contextlib
import ctypes as C
import math
import os
import tempfile

import numpy as np
import torch

from chfem_amd import compute_property, synthetic
from chfem_amd import io as cio
from chfem_amd.guess import LearnedGuess
from chfem_amd.lib import lib, ptr

# local node k of element (row, col, layer) sits at (row + DR, col + DC, layer + DL)
DR = (1, 1, 0, 0, 1, 1, 0, 0)
DC = (0, 1, 1, 0, 0, 1, 1, 0)
DL = (0, 0, 0, 0, 1, 1, 1, 1)
# load cases X, Y, Z, YZ, XZ, XY: axis of the unit gradient, component that has it
AXIS = (0, 1, 2, 1, 2, 1)
COMP = (0, 1, 2, 2, 0, 0)


# ---------------------------------------------------------------------------
# cases
# ---------------------------------------------------------------------------
def listed():
    return [
        # the smallest call: a 32^3 conduction image (Gaussian random field, k
        # 1 / 10), all load cases; set-up, launches and latency
        dict(name="cond_32", kind="property", physics="conductivity", nx=32, ny=32, nz=32, image="grf", contrast=10.0,
             precision="fp64", direction="all", tol=1e-6),
        # a large conduction image with odd edges, mixed precision
        dict(name="cond_odd_large", kind="property", physics="conductivity", nx=233, ny=251, nz=190, image="spheres",
             contrast=50.0, precision="mixed", direction="all", tol=1e-6),
        # a small odd elastic image of three phases with the thermal expansion
        # analysis (a seventh solve)
        dict(name="elas_small_odd", kind="property", physics="elasticity", nx=56, ny=41, nz=37, image="three",
             contrast=10.0, precision="fp64", direction="all", tol=1e-6, alpha=True),
        # an ordinary elastic image, FP64 (the default precision), all load cases
        dict(name="elas_100", kind="property", physics="elasticity", nx=100, ny=100, nz=100, image="spheres",
             contrast=10.0, precision="fp64", direction="all", tol=1e-6),
        # the largest: 256^3 elastic spheres, mixed precision, all load cases
        dict(name="elas_256", kind="property", physics="elasticity", nx=256, ny=256, nz=256, image="spheres",
             contrast=10.0, precision="mixed", direction="all", tol=1e-5),
        # the element-by-element strategy (command line option -p 1), FP64
        dict(name="elas_ebe_96", kind="model", physics="elasticity", nx=96, ny=96, nz=96, image="spheres", contrast=10.0,
             precision="fp64", strategy=1, direction=6, tol=1e-6),
        # a scalar density field (one modulus per voxel), one load case
        dict(name="elas_density_100", kind="density", physics="elasticity", nx=100, ny=100, nz=100, contrast=10.0,
             precision="fp64", direction=1, tol=1e-6),
        # permeability of a thin slab of fibre-like pores, all directions
        dict(name="perm_slab", kind="property", physics="permeability", nx=100, ny=100, nz=10, image="porous",
             porosity=0.6, precision="fp64", direction="all", tol=1e-6, solver="minres"),
        # permeability of a large sphere packing, one direction
        dict(name="perm_160", kind="property", physics="permeability", nx=160, ny=160, nz=160, image="porous",
             porosity=0.35, precision="fp64", direction="z", tol=1e-6, solver="minres"),
        # a batch of small uneven elastic samples, solved together
        dict(name="batch_8", kind="batch", physics="elasticity", samples=8, lo=48, hi=80, contrast=20.0, tol=1e-8),
        # the network's prediction of every load case's field of an image
        dict(name="predict_96", kind="predict", physics="elasticity", nx=96, ny=64, nz=80, contrast=10.0),
        # one training pass (forward, backward) on two 64^3 elastic samples
        dict(name="train_64", kind="train", physics="elasticity", nx=64, ny=64, nz=64, samples=2, contrast=10.0),
    ]


def _edge(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _box(rng, lo, hi):
    n = _edge(rng, lo, hi)
    return dict(zip(("nx", "ny", "nz"), (max(4, int(n * rng.uniform(0.75, 1.3))) for _ in range(3))))


def draw(rng):
    kind = rng.choice(["conductivity", "elasticity", "elasticity", "permeability", "ebe", "density", "batch", "predict",
                       "train"])
    contrast = float(rng.choice([5, 10, 20, 50]))
    precision = rng.choice(["fp64", "mixed"])
    tol = rng.choice([1e-5, 1e-6])
    if kind == "conductivity":
        return dict(kind="property", physics=kind, image=rng.choice(["spheres", "three"]), contrast=contrast,
                    precision=precision, direction=rng.choice(["x", "z", "all"]), tol=tol, **_box(rng, 20, 220))
    if kind == "elasticity":
        return dict(kind="property", physics=kind, image=rng.choice(["spheres", "three"]), contrast=contrast,
                    precision=precision, direction=rng.choice(["x", "yz", "all"]), tol=tol, **_box(rng, 20, 130))
    if kind == "permeability":
        return dict(kind="property", physics=kind, image="porous", porosity=rng.uniform(0.35, 0.6), precision="fp64",
                    direction=rng.choice(["x", "y", "z"]), tol=1e-6, solver=rng.choice(["minres", "minres", "minres3"]),
                    **_box(rng, 24, 120))
    if kind == "ebe":
        return dict(kind="model", physics=rng.choice(["conductivity", "elasticity"]), image=rng.choice(["spheres", "three"]),
                    contrast=contrast, precision=precision, strategy=1, direction=rng.choice([0, 6]), tol=tol,
                    **_box(rng, 20, 90))
    if kind == "density":
        physics = rng.choice(["conductivity", "elasticity"])
        return dict(kind="density", physics=physics, contrast=contrast, precision=precision,
                    direction=rng.choice([0, 1, 2]), tol=tol, **_box(rng, 20, 90))
    if kind == "batch":
        lo = rng.randint(20, 48)
        return dict(kind="batch", physics=rng.choice(["conductivity", "elasticity"]), samples=rng.randint(3, 8), lo=lo,
                    hi=lo + rng.randint(8, 32), contrast=contrast, tol=1e-8)
    return dict(kind=kind, physics=rng.choice(["conductivity", "elasticity"]), samples=2 if kind == "train" else 1,
                contrast=contrast, **{a: 8 * rng.randint(3, 11) for a in ("nx", "ny", "nz")})


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------
def _image(case, seed):
    """uint8 image (z, y, x) of a case."""
    shape = (case["nz"], case["ny"], case["nx"])
    r = max(2.0, min(12.0, min(shape) / 5.0))
    kind = case.get("image", "spheres")
    if kind == "grf":
        return synthetic.grf(shape, sigma=2.0, vf=0.4, seed=seed)
    if kind == "porous":
        return synthetic.porous_spheres(shape, rmin=r / 2, rmax=r, porosity=case["porosity"], seed=seed)[0]
    img = synthetic.spheres(shape, rmin=r / 2, rmax=r, fraction=0.3, seed=seed)
    if kind == "three":
        other = synthetic.spheres(shape, rmin=r / 2, rmax=r, fraction=0.15, seed=seed + 7919)
        img[(other == 255) & (img == 0)] = 128
    img.reshape(-1)[0] = 0
    return img


def _properties(case):
    """{colour: properties} in the order of the model file."""
    c = case.get("contrast", 1.0)
    two = case.get("image") != "three"
    if case["physics"] == "conductivity":
        return {0: 1.0, 255: c} if two else {0: 1.0, 128: math.sqrt(c), 255: c}
    if case["physics"] == "permeability":
        return None
    if two:
        return {0: (1.0, 0.3), 255: (c, 0.2)}
    mats = {0: (1.0, 0.3), 128: (math.sqrt(c), 0.25), 255: (c, 0.2)}
    return {k: v + (a,) for (k, v), a in zip(mats.items(), (2e-5, 1.2e-5, 5e-6))} if case.get("alpha") else mats


ANALYSIS = {"conductivity": 0, "elasticity": 1, "permeability": 2}


class _Files:
    """A model file (and density field) on disk, as a user's program has it."""

    def __init__(self, case, img, props, field=None):
        self.dir = tempfile.TemporaryDirectory(prefix="chfem_case_")
        raw = os.path.join(self.dir.name, "model.raw")
        cio.export_for_chfem(raw, img, ANALYSIS[case["physics"]], props, voxel_size=1.0, export_raw=False,
                             solver_tolerance=case["tol"], solver_maxiter=20000)
        self.nf = raw[:-4] + ".nf"
        self.img = np.ascontiguousarray(img).reshape(-1)
        self.field = None
        if field is not None:
            self.field = os.path.join(self.dir.name, "field.bin")
            field.astype(np.float32).tofile(self.field)


def _density(case, seed):
    """Per-voxel modulus (z, y, x), float32: a smooth random field between 1 and the contrast."""
    rng = np.random.Generator(np.random.PCG64(seed))
    coarse = rng.standard_normal([max(2, n // 8) for n in (case["nz"], case["ny"], case["nx"])])
    out = coarse
    for ax, n in enumerate((case["nz"], case["ny"], case["nx"])):
        at = np.arange(n) * out.shape[ax] / n
        i, f = at.astype(int), at - at.astype(int)
        f = f.reshape([-1 if a == ax else 1 for a in range(3)])
        out = np.take(out, i, ax) * (1 - f) + np.take(out, (i + 1) % out.shape[ax], ax) * f
    out = (out - out.min()) / (out.max() - out.min())
    return (1.0 + (case["contrast"] - 1.0) * out).astype(np.float32)


def _batch_samples(case, seed):
    """[(image, properties)] of a batch."""
    rng = np.random.default_rng(seed)
    out = []
    for s in range(case["samples"]):
        nz, ny, nx = (int(v) for v in rng.integers(case["lo"], case["hi"] + 1, size=3))
        sub = dict(case, nx=nx, ny=ny, nz=nz, image="grf" if case["physics"] == "conductivity" else "spheres")
        out.append((_image(sub, seed * 100 + s), _properties(sub)))
    return out


class _Batch:
    """A batch handle with its samples added (their maps on the GPU)."""

    def __init__(self, case, samples):
        self.case = case
        self.h = lib().chfemBatchCreate()
        self.count = len(samples)
        for img, props in samples:
            f = _Files(case, img, props)
            assert lib().chfemBatchAddSample(self.h, f.nf.encode(), ptr(f.img)) == 1

    def __del__(self):
        if self.h:
            lib().chfemBatchDestroy(self.h)
            self.h = None


SAME, DOWN, UP = 0, 1, 2


def _layers(cout):
    """(mode, inputs, outputs, skip) of the network's layers."""
    return [(SAME, 16, 16, None), (SAME, 16, 16, None), (DOWN, 16, 32, None), (SAME, 32, 32, None), (DOWN, 32, 48, None),
            (SAME, 48, 48, None), (DOWN, 48, 48, None), (SAME, 48, 48, None), (UP, 48, 48, 5), (UP, 48, 32, 3),
            (UP, 32, 16, 1), (SAME, 16, cout, None)]


def _weights(case, seed):
    """Parameters of a network part-way through training: He-scaled weights, small biases."""
    rng = np.random.Generator(np.random.PCG64(seed + 77))
    out = []
    for mode, ci, co, _ in _layers(32 if case["physics"] == "elasticity" else 16):
        n = 8 if mode == DOWN else 27
        out += [rng.standard_normal(co * n * ci) * math.sqrt(2.0 / (n * ci)), 0.05 * rng.standard_normal(co)]
    return np.concatenate(out).astype(np.float32)


def _targets(case, seed):
    """Training samples (image, target): target[v, load * nd + component], smooth fields of order one."""
    nout = 18 if case["physics"] == "elasticity" else 3
    out = []
    for s in range(case["samples"]):
        rng = np.random.Generator(np.random.PCG64(seed * 100 + s))
        small = rng.standard_normal((nout, case["nz"] // 4, case["nx"] // 4, case["ny"] // 4)).astype(np.float32)
        t = small.repeat(4, 1).repeat(4, 2).repeat(4, 3).reshape(nout, -1).T
        out.append((_image(case, seed * 100 + s), np.ascontiguousarray(t)))
    return out


def prepare(case, seed):
    kind = case["kind"]
    props = _properties(case)
    if kind == "property":
        return dict(case=case, img=_image(case, seed), props=props)
    if kind == "model":
        return dict(case=case, files=_Files(case, _image(case, seed), props))
    if kind == "density":
        field = _density(case, seed)
        img = np.zeros(field.shape, np.uint8)
        return dict(case=case, files=_Files(case, img, {0: 1.0} if case["physics"] == "conductivity" else {0: (1.0, 0.3)}, field))
    if kind == "batch":
        return dict(case=case, batch=_Batch(case, _batch_samples(case, seed)))
    net = LearnedGuess("elastic" if case["physics"] == "elasticity" else "thermal")
    net.set_params(_weights(case, seed))
    if kind == "predict":
        return dict(case=case, net=net, img=_image(case, seed), props=props)
    from chfem_amd.guess import element_map, props_vector
    dims = (case["nx"], case["ny"], case["nz"])
    samples = [(element_map(img, props), props_vector(props, net.physics), len(props), dims, t)
               for img, t in _targets(case, seed)]
    return dict(case=case, net=net, samples=samples)


# ---------------------------------------------------------------------------
# one pass
# ---------------------------------------------------------------------------
def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "property":
        more = dict(solver=case["solver"]) if "solver" in case else {}
        rows = compute_property(case["physics"], state["img"], mat_props=state["props"], voxel_size=1.0,
                                solver_tolerance=case["tol"], solver_maxiter=20000, direction=case["direction"],
                                precision=case["precision"], **more)
        n = len(rows[0])
        out = {"C": np.array(rows[:n])}
        if len(rows) > n:
            out["alpha"] = np.array(rows[n])
        return out
    if kind in ("model", "density"):
        f, L = state["files"], lib()
        sdf = f.field.encode() if f.field else None
        if L.hmgInit(f.nf.encode(), None, sdf, ptr(f.img)) != 1:
            raise RuntimeError("hmgInit failed")
        try:
            L.hmgSetParallelStrategyFlag(case.get("strategy", 0))
            L.hmgSetPrecisionFlag(1 if case["precision"] == "mixed" else 0)
            L.hmgSetHomogenizationFlag(case["direction"])
            n = 6 if case["physics"] == "elasticity" else 3
            Cm = np.zeros((n, n))
            if L.hmgPrepare() != 1 or L.hmgSolveResident(ptr(Cm)) != 1:
                raise RuntimeError("the homogenization failed")
            L.hmgRelease()
        finally:
            L.hmgSetParallelStrategyFlag(0)
            L.hmgSetPrecisionFlag(0)
            L.hmgEnd()
        return {"C": Cm}
    if kind == "batch":
        b = state["batch"]
        if lib().chfemBatchSolve(b.h, case["tol"], 20000) == 0:
            raise RuntimeError("chfemBatchSolve failed")
        n = 6 if case["physics"] == "elasticity" else 3
        out = [np.zeros((n, n)) for _ in range(b.count)]
        for k, Cm in enumerate(out):
            lib().chfemBatchGetC(b.h, k, ptr(Cm))
        return out
    net = state["net"]
    if kind == "predict":
        return net.predict(state["img"], state["props"])
    net.zero_gradients()
    for s in state["samples"]:
        net.accumulate(s)
    return {"gradients": net.gradients()}


def work(case):
    """Bytes and operations of one pass.  A homogenization: the CG or MINRES
    iterations such an image takes (an estimate from its longest edge), each
    with one operator application and the vectors a Krylov iteration streams
    (residual, direction and iterate, 5 passes); the voxels read once."""
    kind = case["kind"]
    el = case["physics"] == "elasticity"
    if kind in ("predict", "train"):
        v = case["nx"] * case["ny"] * case["nz"]
        flops, at = 0.0, v
        for mode, ci, co, _ in _layers(32 if el else 16):
            at = at // 8 if mode == DOWN else at * 8 if mode == UP else at
            flops += 2.0 * at * ci * co * (8 if mode == DOWN else 27)
        nout = 18 if el else 3
        if kind == "predict":
            return {"bytes": v * (2.0 + 4 * nout), "flops": flops}
        return {"bytes": case["samples"] * v * (2.0 + 4 * nout), "flops": 3 * flops * case["samples"]}

    def solve(n, edge, loads, w):
        digits = -math.log10(case["tol"]) / 6
        nd = 3 if el else 1
        if case["physics"] == "permeability":
            pore = case["porosity"]
            its, n, nd, per = 6.0 * edge * digits, n * pore, 4, 250
        else:
            its, per = (4.3 if el else 2.5) * edge * digits, 190 if el else 50
        return its * loads * n * (5.0 * nd * w + 1), its * loads * n * (per + 10 * nd), n

    if kind == "batch":
        n = ((case["lo"] + case["hi"]) / 2.0)
        b, f, _ = solve(n ** 3, n, 6 if el else 3, 4)
        return {"bytes": case["samples"] * b, "flops": case["samples"] * f}
    every = case["direction"] in ("all", 6)
    loads = (6 if el else 3) if every else 1
    n = case["nx"] * case["ny"] * case["nz"]
    b, f, _ = solve(n, max(case["nx"], case["ny"], case["nz"]), loads, 4 if case["precision"] == "mixed" else 8)
    return {"bytes": b + n, "flops": f}


# ---------------------------------------------------------------------------
# the same in plain torch, 64 bits
# ---------------------------------------------------------------------------
def _device():
    return torch.device("cuda" if torch.cuda.is_available() else "cpu")


def _integral(i, j, p, q, flip):
    """Integral over the unit voxel of d_p N_i d_q N_j (-1: no derivative)."""
    a, b = _corner(i, flip), _corner(j, flip)
    v = 1.0
    for t in range(3):
        si, sj = (1.0 if a[t] else -1.0), (1.0 if b[t] else -1.0)
        if t == p and t == q:
            v *= si * sj
        elif t == p:
            v *= 0.5 * si
        elif t == q:
            v *= 0.5 * sj
        else:
            v *= 1.0 / 3.0 if a[t] == b[t] else 1.0 / 6.0
    return v


def _corner(k, flip):
    """Corner of local node k in the voxel's frame: x along columns, y against
    rows, z against layers (Stokes: along layers)."""
    return DC[k], 1 - DR[k], DL[k] if flip else 1 - DL[k]


def _unit_matrices(physics, flip=False):
    """Unit-voxel matrices: conduction (one), elasticity (lambda and mu parts)."""
    lap = np.array([[sum(_integral(i, j, a, a, flip) for a in range(3)) for j in range(8)] for i in range(8)])
    if physics == "conductivity":
        return [lap]
    kl, km = np.zeros((24, 24)), np.zeros((24, 24))
    for i in range(8):
        for j in range(8):
            for a in range(3):
                for b in range(3):
                    kl[3 * i + a, 3 * j + b] = _integral(i, j, a, b, flip)
                    km[3 * i + a, 3 * j + b] = _integral(i, j, b, a, flip) + (lap[i, j] if a == b else 0.0)
    return [kl, km]


def _lame(E, nu):
    return E * nu / ((1 + nu) * (1 - 2 * nu)), E / (2 * (1 + nu))


class _Periodic:
    """Periodic voxel problem sum_j c_j(e) K_j on a (layer, column, row) grid,
    solved by CG with the mean medium inverted in Fourier space."""

    def __init__(self, physics, coef):
        self.dev = coef[0].device
        self.nd = 3 if physics == "elasticity" else 1
        self.coef = coef  # [element fields]
        self.shape = coef[0].shape
        self.n = coef[0].numel()
        mats = _unit_matrices(physics)
        self.K = torch.tensor(np.concatenate(mats), dtype=torch.float64, device=self.dev)
        self.corner = np.array([_corner(k, False) for k in range(8)], dtype=float)
        self._precondition(sum(float(c.mean()) * m for c, m in zip(coef, mats)))

    def gather(self, u):
        """(8 nd, n) nodal values of every element of u (nd, grid)."""
        U = torch.empty((8, self.nd) + tuple(self.shape), dtype=torch.float64, device=self.dev)
        for k in range(8):
            U[k] = torch.roll(u, (-DL[k], -DC[k], -DR[k]), (1, 2, 3))
        return U.view(8 * self.nd, self.n)

    def scatter(self, F):
        F = F.view((8, self.nd) + tuple(self.shape))
        out = torch.zeros((self.nd,) + tuple(self.shape), dtype=torch.float64, device=self.dev)
        for k in range(8):
            out += torch.roll(F[k], (DL[k], DC[k], DR[k]), (1, 2, 3))
        return out

    def forces(self, U):
        ke = 8 * self.nd
        F = self.K @ U
        out = F[:ke] * self.coef[0].view(1, -1)
        if len(self.coef) > 1:
            out += F[ke:] * self.coef[1].view(1, -1)
        return out

    def apply(self, u):
        return self.scatter(self.forces(self.gather(u)))

    def _precondition(self, K0):
        nz, nx, ny = self.shape
        f = [torch.fft.fftfreq(nz, dtype=torch.float64, device=self.dev).view(-1, 1, 1),
             torch.fft.fftfreq(nx, dtype=torch.float64, device=self.dev).view(1, -1, 1),
             torch.fft.rfftfreq(ny, dtype=torch.float64, device=self.dev).view(1, 1, -1)]
        P = torch.stack([torch.exp(2j * math.pi * (f[0] * DL[k] + f[1] * DC[k] + f[2] * DR[k])) for k in range(8)])
        grid = P.shape[1:]
        P = P.reshape(8, -1)
        nd = self.nd
        K0 = torch.tensor(K0, dtype=torch.complex128, device=self.dev).view(8, nd, 8, nd)
        M = [[None] * nd for _ in range(nd)]
        for a in range(nd):
            for b in range(nd):
                M[a][b] = (P.conj() * (K0[:, a, :, b].contiguous() @ P)).sum(0)
        if nd == 1:
            d = M[0][0].real
            d[0] = 1.0
            inv = 1.0 / d
            inv[0] = 0.0
            self.inv = [[inv.view(grid)]]
            return
        # inverse of the 3 x 3 Hermitian symbol by cofactors
        co = [[M[(i + 1) % 3][(j + 1) % 3] * M[(i + 2) % 3][(j + 2) % 3] - M[(i + 1) % 3][(j + 2) % 3] * M[(i + 2) % 3][(j + 1) % 3]
               for j in range(3)] for i in range(3)]
        det = sum(M[0][j] * co[0][j] for j in range(3)).real
        det[0] = 1.0
        s = 1.0 / det
        s[0] = 0.0
        self.inv = [[(co[j][i] * s).view(grid) for j in range(3)] for i in range(3)]

    def precond(self, r):
        h = torch.fft.rfftn(r, dim=(1, 2, 3))
        g = torch.stack([sum(self.inv[a][b] * h[b] for b in range(self.nd)) for a in range(self.nd)])
        return torch.fft.irfftn(g, s=tuple(self.shape), dim=(1, 2, 3))

    def solve(self, b, tol=1e-11, maxit=400):
        x = torch.zeros_like(b)
        r = b.clone()
        z = self.precond(r)
        d = z.clone()
        rz = rz0 = float((r * z).sum())
        for _ in range(maxit):
            if not rz > tol * tol * rz0:
                break
            q = self.apply(d)
            a = rz / float((d * q).sum())
            x += a * d
            r -= a * q
            z = self.precond(r)
            rz, old = float((r * z).sum()), rz
            d = z + (rz / old) * d
        return x

    def ramp(self, load):
        """Nodal values of the unit gradient of a load case within an element."""
        comp = COMP[load] if self.nd == 3 else 0
        R = np.zeros(8 * self.nd)
        R[comp::self.nd] = self.corner[:, AXIS[load]]
        return torch.tensor(R, dtype=torch.float64, device=self.dev)

    def gradient_mean(self, u, weight):
        """(nd, 3): sum over elements of weight * mean gradient of u."""
        out = np.zeros((self.nd, 3))
        for k in range(8):
            uk = torch.roll(u, (-DL[k], -DC[k], -DR[k]), (1, 2, 3)) * weight
            s = uk.sum((1, 2, 3)).cpu().numpy()
            for a in range(3):
                out[:, a] += (0.25 if self.corner[k, a] else -0.25) * s
        return out

    def column(self, load):
        """Column of the effective matrix for a load case."""
        R = self.ramp(load)
        ke = 8 * self.nd
        f = self.K @ R
        F = f[:ke].view(-1, 1) * self.coef[0].reshape(1, -1)
        if len(self.coef) > 1:
            F = F + f[ke:].view(-1, 1) * self.coef[1].reshape(1, -1)
        u = self.solve(-self.scatter(F))
        del F
        G = []
        for c in self.coef:
            g = self.gradient_mean(u, c)
            g[COMP[load] if self.nd == 3 else 0, AXIS[load]] += float(c.sum())
            G.append(g / self.n)
        return self.flux(G)

    def flux(self, G):
        if self.nd == 1:
            return G[0][0]
        tr, m = np.trace(G[0]), G[1] + G[1].T
        return np.array([tr + m[0, 0], tr + m[1, 1], tr + m[2, 2], m[1, 2], m[0, 2], m[0, 1]])

    def expansion(self, Cm, stress):
        """Effective thermal expansion for the thermal stress (D alpha)_xx of every element."""
        f = np.zeros((24, 1))
        for k in range(8):
            for a in range(3):
                f[3 * k + a, 0] = 0.25 if self.corner[k, a] else -0.25
        F = torch.tensor(f, dtype=torch.float64, device=self.dev) * stress.reshape(1, -1)
        u = self.solve(self.scatter(F))
        mean = self.flux([self.gradient_mean(u, c) / self.n for c in self.coef])
        beta = -mean
        beta[:3] += float(stress.mean())
        return np.linalg.solve(Cm, beta)


def _element_map(img, colours):
    lut = np.zeros(256, dtype=np.int64)
    for i, c in enumerate(colours):
        lut[c] = i
    return torch.tensor(np.ascontiguousarray(lut[img].transpose(0, 2, 1)), device=_device())


def _effective(physics, img, props, loads):
    em = _element_map(img, list(props))
    table = [(float(p),) if physics == "conductivity" else _lame(*p[:2]) for p in props.values()]
    coef = [torch.tensor([t[j] for t in table], dtype=torch.float64, device=em.device)[em] for j in range(len(table[0]))]
    P = _Periodic(physics, coef)
    n = 6 if physics == "elasticity" else 3
    Cm = np.zeros((n, n))
    for d in loads:
        Cm[:, d] = P.column(d)
    return Cm, P, em


def _stokes(img, loads, tol=1e-11, maxit=20000):
    """Permeability columns: stabilised trilinear Stokes flow in the pore voxels, by MINRES."""
    dev = _device()
    pore = torch.tensor(np.ascontiguousarray((img == 0).transpose(0, 2, 1)), device=dev)
    around = torch.zeros(pore.shape, dtype=torch.int64, device=dev)
    for k in range(8):
        around += torch.roll(pore.long(), (DL[k], DC[k], DR[k]), (0, 1, 2))
    mask = torch.stack([around == 8] * 3 + [around > 0]).double()
    lap = _unit_matrices("conductivity", True)[0]
    K = np.zeros((8, 4, 8, 4))
    K[:, :3, :, :3] = _unit_matrices("elasticity", True)[1].reshape(8, 3, 8, 3)
    for i in range(8):
        for j in range(8):
            for a in range(3):
                g = _integral(i, j, a, -1, True)
                K[i, a, j, 3] = g
                K[j, 3, i, a] = g
    K[:, 3, :, 3] = -lap / 6.0
    # pore elements only: their nodes, compacted
    l, c, r = torch.nonzero(pore, as_tuple=True)
    nz, nx, ny = pore.shape
    N = pore.numel()
    node = torch.stack([(r + DR[k]) % ny + ((c + DC[k]) % nx) * ny + ((l + DL[k]) % nz) * nx * ny for k in range(8)])
    used, at = torch.unique(node, return_inverse=True)
    mask = mask.view(4, N)[:, used]
    # neighbours: of every node, the element for which it is local node k
    elem_of = torch.full((8, used.numel()), pore.sum().item(), dtype=torch.int64, device=dev)
    for k in range(8):
        elem_of[k, at[k]] = torch.arange(at.shape[1], device=dev)
    Kt = torch.tensor(K.reshape(32, 32), device=dev)
    Ne = at.shape[1]
    F = torch.zeros((8, 4, Ne + 1), dtype=torch.float64, device=dev)

    def apply(v):
        U = torch.stack([v[:, at[k]] for k in range(8)]).view(32, Ne)
        F[:, :, :Ne] = (Kt @ U).view(8, 4, Ne)
        out = F[0][:, elem_of[0]]
        for k in range(1, 8):
            out += F[k][:, elem_of[k]]
        return out * mask

    count = around.reshape(-1)[used].double()
    diag = torch.stack([count * K[0, a, 0, a] for a in range(3)] + [count * (lap[0, 0] / 6.0)])
    minv = mask / diag
    Cm = np.zeros((3, 3))
    for d in loads:
        b = torch.zeros_like(mask)
        b[d] = mask[d]
        # preconditioned conjugate residuals (MINRES for the definite preconditioner)
        x = torch.zeros_like(b)
        z = minv * b
        s = apply(z)
        p, q = z.clone(), s.clone()
        zs, z0 = float((z * s).sum()), float((b * z).sum())
        res = b.clone()
        for it in range(maxit):
            mq = minv * q
            a = zs / float((q * mq).sum())
            x += a * p
            z -= a * mq
            res -= a * q
            if float((res * z).sum()) <= tol * tol * z0:
                break
            s = apply(z)
            zs, old = float((z * s).sum()), zs
            p = z + (zs / old) * p
            q = s + (zs / old) * q
        Cm[:, d] = (x[:3].sum(1) / N).cpu().numpy()
    return Cm


def _shift(x, d):
    return torch.roll(x, [-v for v in d], (0, 1, 2))


def _conv(mode, x, W):
    co, taps, ci = W.shape
    out = 0
    if mode == DOWN:
        for t in range(8):
            out = out + x[t >> 2::2, (t >> 1) & 1::2, t & 1::2] @ W[:, t].T
        return out
    if mode == UP:
        x = x.repeat_interleave(2, 0).repeat_interleave(2, 1).repeat_interleave(2, 2)
    for t in range(27):
        out = out + _shift(x, (t // 9 - 1, (t // 3) % 3 - 1, t % 3 - 1)) @ W[:, t].T
    return out


def _network(case, w, img):
    """Prediction (voxels, outputs) of the network with parameters w."""
    props = _properties(case)
    el = case["physics"] == "elasticity"
    first = np.array([p[0] if el else p for p in props.values()])
    tab = np.zeros((len(props), 16))
    tab[:, 0] = np.log10(first / first.max())
    if el:
        tab[:, 1] = [(p[1] - 0.25) * 4.0 for p in props.values()]
    em = _element_map(img, list(props))
    x = torch.tensor(tab, device=em.device)[em]
    at, acts = 0, []
    layers = _layers(32 if el else 16)
    for k, (mode, ci, co, skip) in enumerate(layers):
        n = co * (8 if mode == DOWN else 27) * ci
        W, b = w[at:at + n].view(co, -1, ci), w[at + n:at + n + co]
        at += n + co
        x = _conv(mode, x, W) + b
        if skip is not None:
            x = x + acts[skip]
        if k + 1 < len(layers):
            x = torch.relu(x)
        acts.append(x)
    return x[..., :18 if el else 3].reshape(em.numel(), -1)


def exact(case, seed):
    kind, physics = case["kind"], case["physics"]
    n = 6 if physics == "elasticity" else 3
    names = {"x": [0], "y": [1], "z": [2], "yz": [3], "xz": [4], "xy": [5], "all": range(n), 6: range(n)}
    with contextlib.suppress(RuntimeError):
        torch.backends.cuda.matmul.allow_tf32 = False
    if kind == "property" and physics == "permeability":
        return {"C": _stokes(_image(case, seed), names[case["direction"]])}
    if kind in ("property", "model"):
        loads = names.get(case["direction"], [case["direction"]])
        props = _properties(case)
        Cm, P, em = _effective(physics, _image(case, seed), props, loads)
        out = {"C": Cm}
        if case.get("alpha"):
            da = [(3 * lam + 2 * mu) * p[2] for p in props.values() for lam, mu in [_lame(*p[:2])]]
            out["alpha"] = P.expansion(Cm, torch.tensor(da, device=em.device)[em])
        return out
    if kind == "density":
        v = _density(case, seed).astype(np.float64)
        lo, hi = v.min(), v.max()
        q = np.floor(65535 * (v - lo) / (hi - lo))
        s = torch.tensor(np.ascontiguousarray((q / 65535 * (hi - lo) + lo).transpose(0, 2, 1)), device=_device())
        P = _Periodic(physics, [s] if physics == "conductivity" else [c * s for c in _lame(1.0, 0.3)])
        Cm = np.zeros((n, n))
        for d in names.get(case["direction"], [case["direction"]]):
            Cm[:, d] = P.column(d)
        return {"C": Cm}
    if kind == "batch":
        return [_effective(physics, img, props, range(n))[0] for img, props in _batch_samples(case, seed)]
    w = torch.tensor(_weights(case, seed), dtype=torch.float64, device=_device())
    if kind == "predict":
        with torch.no_grad():
            return _network(case, w, _image(case, seed)).cpu().numpy()
    w.requires_grad_(True)
    for img, t in _targets(case, seed):
        y = _network(case, w, img)
        ((y - torch.tensor(t, dtype=torch.float64, device=w.device)) ** 2).mean().backward()
    return {"gradients": w.grad.cpu().numpy()}
