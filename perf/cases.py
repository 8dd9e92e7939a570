"""Performance cases: what programs that use this package ask of it, over the range of sizes it is used at.

Each case names a kind of work and its sizes:

* ``call``      one complete ``homogenize`` call on host labels (validation, upload, set-up, solve, certificate);
* ``batch``     one ``homogenize_batch`` call over cells of uneven size;
* ``operator``  K u on the six load cases of a resident cell;
* ``precond``   the Green preconditioner on the six load cases of a resident cell;
* ``protocol``  the node-major FP64 operator protocol (K u, then M r) a caller's own iteration uses;
* ``recover``   right-hand sides and element-centre fields of six displacement fields;
* ``simp``      one design iteration: C_eff of a density field and its gradient.

Cells are seeded: thresholded random fields (two-phase media such as digital rocks), random spheres, periodic Voronoi
polycrystals and the analytic weave.  ``exact`` computes the same outputs in FP64 with plain torch.
"""
import math
import sys
from pathlib import Path

import numpy as np
import torch

_ROOT = Path(__file__).resolve().parents[1]
for _p in (_ROOT / "voxel-lmfem_amd", _ROOT):
    if str(_p) not in sys.path:
        sys.path.insert(0, str(_p))

PAIRS = [(i, j) for i in range(6) for j in range(i, 6)]


def _call(cell, nx, ny, nz, precision, **more):
    return dict(kind="call", cell=cell, nx=nx, ny=ny, nz=nz, precision=precision, **more)


def listed():
    return [
        # Parameter studies and screening solve very small cells one after the other: launches and host work count.
        dict(_call("rock", 21, 25, 18, "mixed"), name="call_small_21x25x18"),
        # The 32^3 random-sphere cell in FP64, the smallest configured workload.
        dict(_call("spheres", 32, 32, 32, "fp64"), name="call_spheres_32_fp64"),
        # A sub-volume cut from a scan: axes of arbitrary length (3*37, 2*47, 2*59), slices thicker than pixels.
        dict(_call("rock", 111, 94, 118, "mixed", dz=1.5), name="call_crop_111x94x118"),
        # The woven composite cell with per-voxel tow frames, voxels not cubic.
        dict(_call("weave", 128, 128, 128, "mixed"), name="call_weave_128"),
        # A two-phase medium solved entirely in FP64.
        dict(_call("rock", 160, 160, 160, "fp64"), name="call_rock_160_fp64"),
        # The 256^3, 200-grain polycrystal: the largest ordinary cell.
        dict(_call("grains", 256, 256, 256, "mixed", grains=200), name="call_grains_256"),
        # Many statistical volume elements of uneven size in one call.
        dict(kind="batch", edges="32,48,27,64,32,40,48,32,50,64,36,32", name="batch_uneven_12"),
        # One operator and one preconditioner step of a caller's own iteration on a small cell.
        dict(kind="protocol", nx=40, ny=36, nz=44, name="protocol_40x36x44"),
        # The FP32 operator on six load cases of an ordinary polycrystal.
        dict(kind="operator", cell="grains", nx=192, ny=160, nz=144, grains=120, dtype="float32",
             name="operator_192x160x144_f32"),
        # The FP32 preconditioner on six load cases, axes of 2^a 3^b 5^c.
        dict(kind="precond", nx=150, ny=100, nz=125, dtype="float32", name="precond_150x100x125_f32"),
        # Post-processing: right-hand sides and centre fields of six loads.
        dict(kind="recover", cell="grains", nx=110, ny=96, nz=100, grains=60, name="recover_110x96x100"),
        # Topology optimisation: one forward and backward pass over a density field.
        dict(kind="simp", nx=40, ny=40, nz=40, name="simp_40"),
    ]


def _size(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _grid(rng, lo, hi, most):
    while True:
        n = [_size(rng, lo, hi) for _ in range(3)]
        if n[0] * n[1] * n[2] <= most:
            return dict(nx=n[0], ny=n[1], nz=n[2])


def draw(rng):
    kind = rng.choice(["call"] * 8 + ["operator"] * 3 + ["precond"] * 3 + ["protocol", "protocol", "batch", "recover",
                                                                        "simp"])
    if kind == "call":
        precision = rng.choice(["mixed", "mixed", "fp64"])
        cell = rng.choice(["rock", "rock", "grains", "grains", "spheres", "weave"])
        if cell == "weave":
            n = _size(rng, 40, 128)
            return _call(cell, n, n, n, precision)
        if cell == "spheres":
            n = _size(rng, 16, 96)
            return _call(cell, n, n, n, precision)
        g = _grid(rng, 16, 176, 2_500_000)
        more = dict(grains=rng.randint(8, 250)) if cell == "grains" else dict(dz=rng.choice([1.0, 1.0, 1.5, 2.5]))
        return _call(cell, g["nx"], g["ny"], g["nz"], precision, **more)
    if kind == "batch":
        edges = [_size(rng, 16, 72) for _ in range(rng.randint(4, 10))]
        return dict(kind="batch", edges=",".join(str(e) for e in edges))
    if kind == "operator":
        return dict(kind=kind, cell=rng.choice(["grains", "rock"]), grains=rng.randint(8, 250),
                    dtype=rng.choice(["float32", "float32", "float64"]), **_grid(rng, 16, 256, 6_000_000))
    if kind == "precond":
        return dict(kind=kind, dtype=rng.choice(["float32", "float32", "float64"]), **_grid(rng, 16, 256, 6_000_000))
    if kind == "protocol":
        return dict(kind=kind, **_grid(rng, 12, 96, 500_000))
    if kind == "recover":
        return dict(kind=kind, cell="grains", grains=rng.randint(8, 250), **_grid(rng, 16, 160, 1_500_000))
    n = _size(rng, 16, 40)
    return dict(kind="simp", nx=n, ny=n, nz=n)


# ---- seeded cells ---------------------------------------------------------------

def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed))


def _smooth_field(shape, seed, sigma):
    """Periodic Gaussian random field (nz, ny, nx) with correlation length sigma voxels."""
    f = torch.randn(shape, generator=_gen(seed), device="cuda", dtype=torch.float32)
    k2 = sum((torch.fft.fftfreq(n, device="cuda")[(slice(None),) + (None,) * (2 - a)]) ** 2 for a, n in enumerate(shape))
    return torch.fft.ifftn(torch.fft.fftn(f) * torch.exp(-2.0 * (math.pi * sigma) ** 2 * k2)).real


def _rock(shape, seed, fraction=0.3):
    f = _smooth_field(shape, seed, 2.5).reshape(-1)
    cut = torch.sort(f).values[int(f.numel() * (1.0 - fraction))]
    return (f > cut).to(torch.uint8).reshape(shape)


def _grains(shape, seed, count):
    """Periodic Voronoi labels (nearest seed point by the minimum image)."""
    nz, ny, nx = shape
    p = torch.rand(count, 3, generator=_gen(seed), device="cuda")
    best = torch.full(shape, float("inf"), device="cuda")
    label = torch.zeros(shape, dtype=torch.int32, device="cuda")
    sq = []
    for a, n in enumerate(shape):
        d = torch.arange(n, device="cuda") + 0.5 - p[:, a:a + 1] * n
        d = d - n * torch.round(d / n)
        sq.append(d * d)
    for g in range(count):
        d = sq[0][g][:, None, None] + sq[1][g][None, :, None] + sq[2][g][None, None, :]
        near = d < best
        label.masked_fill_(near, g)
        best = torch.where(near, d, best)
    return label


def _rotations(count, rng):
    q = rng.normal(size=(count, 4))
    q /= np.linalg.norm(q, axis=1, keepdims=True)
    w, x, y, z = q.T
    return np.stack([1 - 2 * (y * y + z * z), 2 * (x * y - w * z), 2 * (x * z + w * y),
                     2 * (x * y + w * z), 1 - 2 * (x * x + z * z), 2 * (y * z - w * x),
                     2 * (x * z - w * y), 2 * (y * z + w * x), 1 - 2 * (x * x + y * y)], axis=1).reshape(-1, 3, 3)


def _bond(R):
    """Stress rotation matrices T (k, 6, 6) of R (k, 3, 3), order 11, 22, 33, 23, 13, 12: C' = T C T^T."""
    a, b = [0, 1, 2, 1, 0, 0], [0, 1, 2, 2, 2, 1]
    T = R[:, a][:, :, a] * R[:, b][:, :, b]
    T[:, :, 3:] = T[:, :, 3:] + (R[:, a][:, :, b] * R[:, b][:, :, a])[:, :, 3:]
    return T


def _cubic(C11, C12, C44):
    C = np.zeros((6, 6))
    C[:3, :3] = C12
    C[range(3), range(3)] = C11
    C[range(3, 6), range(3, 6)] = C44
    return C


def _isotropic(E, nu):
    lam, mu = E * nu / ((1 + nu) * (1 - 2 * nu)), E / (2 * (1 + nu))
    return _cubic(lam + 2 * mu, lam, mu)


def _orthotropic(m):
    S = np.zeros((6, 6))
    S[0, 0], S[1, 1], S[2, 2] = 1 / m["E1"], 1 / m["E2"], 1 / m["E3"]
    S[0, 1] = S[1, 0] = -m["nu12"] / m["E1"]
    S[0, 2] = S[2, 0] = -m["nu13"] / m["E1"]
    S[1, 2] = S[2, 1] = -m["nu23"] / m["E2"]
    S[3, 3], S[4, 4], S[5, 5] = 1 / m["G23"], 1 / m["G13"], 1 / m["G12"]
    return np.linalg.inv(S)


def _two_phase(rng, lo=5.0, hi=25.0):
    E = 10.0 ** rng.uniform(math.log10(lo), math.log10(hi))
    return {0: dict(kind="isotropic", E=3.0, nu=0.35), 1: dict(kind="isotropic", E=3.0 * E, nu=0.22)}


def _weave(n, seed):
    """The analytic weave, shifted in the plane and with yarn moduli varied by the seed."""
    from voxel_lmfem.cells import reference_weave
    (phase, materials, domain, orientation), _ = reference_weave(n)
    rng = np.random.default_rng(seed)
    shift = (0, int(rng.integers(n)), int(rng.integers(n)))
    roll = lambda a: np.ascontiguousarray(np.roll(a, shift, axis=(0, 1, 2)))  # noqa: E731
    materials[1] = dict(materials[1], E1=float(rng.uniform(1.2e5, 1.5e5)), G12=float(rng.uniform(4.5e3, 5.5e3)))
    return roll(phase), materials, domain, {k: roll(v) for k, v in orientation.items()}


def _cell(case, seed):
    """(labels on the GPU or host, materials, domain, orientation) of a cell."""
    rng = np.random.default_rng(seed)
    shape = (case["nz"], case["ny"], case["nx"])
    domain = np.array([case["nx"], case["ny"], case["nz"] * case.get("dz", 1.0)], dtype=float) / case["nx"]
    if case["cell"] == "rock":
        return _rock(shape, seed), _two_phase(rng), domain, None
    if case["cell"] == "grains":
        C = _cubic(168.4, 121.4, 75.4)
        T = _bond(_rotations(case["grains"], rng))
        rotated = T @ C @ T.transpose(0, 2, 1)
        rotated = 0.5 * (rotated + rotated.transpose(0, 2, 1))
        return _grains(shape, seed, case["grains"]), {g: dict(kind="anisotropic", C=rotated[g])
                                                      for g in range(case["grains"])}, domain, None
    if case["cell"] == "spheres":
        from voxel_lmfem.cells import periodic_spheres
        (phase, _, domain, _), _ = periodic_spheres(case["nx"], radius=3.0, fraction=0.30, seed=seed)
        return phase, _two_phase(rng, 20.0, 25.0), domain, None
    return _weave(case["nx"], seed)


def _host(labels):
    return labels.cpu().numpy() if isinstance(labels, torch.Tensor) else labels


def _batch_cells(case, seed):
    from voxel_lmfem.cells import periodic_spheres
    cells, rng = [], np.random.default_rng(seed)
    for k, n in enumerate(int(e) for e in case["edges"].split(",")):
        (phase, _, domain, _), _ = periodic_spheres(n, radius=float(rng.integers(2, 6)),
                                                    fraction=float(rng.uniform(.1, .4)), seed=seed * 100 + k)
        cells.append((phase, _two_phase(rng, 5.0, 50.0), domain))
    return cells


def _density(case, seed):
    f = _smooth_field((case["nz"], case["ny"], case["nx"]), seed, 3.0)
    return 0.05 + 0.95 * (f - f.min()) / (f.max() - f.min())


def _randn(shape, seed, dtype):
    return torch.randn(shape, generator=_gen(seed), device="cuda", dtype=getattr(torch, dtype))


def _resident(case, seed):
    """Cell handle over labels that are already on the GPU."""
    from voxel_lmfem.gpu import Cell
    from voxel_lmfem.materials import build_field_device
    labels, materials, domain, _ = _cell(case, seed)
    labels = torch.as_tensor(labels, device="cuda")
    field = build_field_device(labels.to(torch.int32), materials)
    shape = tuple(labels.shape)
    return Cell(field, shape, domain / np.array(shape[::-1], dtype=float))


_MEDIUM = dict(lam=60.0, mu=40.0)
_ONE = {0: dict(kind="isotropic", E=100.0, nu=0.3)}


def _plain_cell(case):
    """A uniform cell for the preconditioner alone, which depends on grid and voxel size only."""
    from voxel_lmfem.gpu import Cell
    from voxel_lmfem.materials import build_field_device
    shape = (case["nz"], case["ny"], case["nx"])
    return Cell(build_field_device(torch.zeros(shape, dtype=torch.int32, device="cuda"), _ONE), shape,
                (1.0 / case["nx"],) * 3)


def prepare(case, seed):
    kind, st = case["kind"], {"case": case}
    if kind == "call":
        labels, materials, domain, orientation = _cell(case, seed)
        st.update(labels=_host(labels), materials=materials, domain=domain, orientation=orientation)
    elif kind == "batch":
        st.update(cells=_batch_cells(case, seed))
    elif kind == "simp":
        rho = _density(case, seed)
        st.update(rho=rho.requires_grad_(True), weights=torch.zeros(6, 6, dtype=torch.float64))
        st["weights"][0, 0] = 1.0
        st["weights"][:3, :3] += 1.0 / 9.0
    else:
        n = case["nx"] * case["ny"] * case["nz"]
        if kind == "precond":
            from voxel_lmfem.gpu import Preconditioner
            cell = _plain_cell(case)
            st.update(cell=cell, u=_randn((6, 3, n), seed, case["dtype"]),
                      precond=Preconditioner(cell, _MEDIUM["lam"], _MEDIUM["mu"], precision=case["dtype"], nrhs_max=6))
        elif kind == "protocol":
            cell = _resident(dict(case, cell="grains", grains=20), seed)
            cell.enable_preconditioner(_MEDIUM["lam"], _MEDIUM["mu"], precision="float64")
            st.update(cell=cell, u=_randn((1, 3 * n), seed, "float64"), r=_randn((1, 3 * n), seed + 1, "float64"))
        elif kind == "operator":
            st.update(cell=_resident(case, seed), u=_randn((6, 3, n), seed, case["dtype"]))
        else:
            st.update(cell=_resident(case, seed), u=_randn((6, 3, n), seed, "float64").mul_(1e-3), macro=np.eye(6))
    return st


def run(st):
    case = st["case"]
    kind = case["kind"]
    if kind == "call":
        from voxel_lmfem import homogenize
        out = homogenize(st["labels"], st["materials"], st["domain"], orientation=st["orientation"], backend="gpu",
                         precision=case["precision"])
        return np.array(out["CH"])
    if kind == "batch":
        from voxel_lmfem.solver import homogenize_batch
        return [np.array(r["CH"]) for r in homogenize_batch(st["cells"], autotune=False)]
    if kind == "simp":
        from voxel_lmfem.adjoint import density_ceff
        st["rho"].grad = None
        C = density_ceff(st["rho"], (1.0, 1.0, 1.0))
        (st["weights"] * C).sum().backward()
        return dict(C=C.detach(), grad=st["rho"].grad)
    cell = st["cell"]
    if kind == "operator":
        return cell.apply_planes(st["u"])
    if kind == "precond":
        return st["precond"].apply_planes(st["u"])
    if kind == "protocol":
        return cell.apply(st["u"]), cell.apply_precond(st["r"])
    strain, stress, energy = cell.center_fields_planes(st["u"], st["macro"])
    return cell.rhs_planes(st["macro"]), strain, stress, energy


# Iterations a solve of each cell takes, in round numbers: its least work is that many operator and preconditioner
# steps.
_ITERATIONS = dict(rock=30, spheres=45, grains=15, weave=55)


def _solve_work(n, iterations, size):
    """Per iteration and load: p read and q written, r read and z written (3 entries of `size` bytes a node); the
    strain modes of the element and three complex-from-real transforms."""
    return dict(bytes=n * 6 * iterations * 12 * size, flops=n * 6 * iterations * (500 + 15 * math.log2(n)))


def work(case):
    kind = case["kind"]
    if kind == "batch":
        each = [_solve_work(int(e) ** 3, 60, 4) for e in case["edges"].split(",")]
        return {k: sum(w[k] for w in each) for k in ("bytes", "flops")}
    n = case["nx"] * case["ny"] * case["nz"]
    if kind == "call":
        return _solve_work(n, _ITERATIONS[case["cell"]], 4 if case["precision"] == "mixed" else 8)
    if kind == "simp":
        return _solve_work(n, 400, 8)
    if kind == "protocol":
        return dict(bytes=n * 4 * 24, flops=n * (500 + 15 * math.log2(n)))
    if kind == "recover":
        return dict(bytes=n * 6 * 8 * (3 + 3 + 13), flops=n * 6 * 250)
    size = 8 if case["dtype"] == "float64" else 4
    flops = 500 if kind == "operator" else 15 * math.log2(n)
    return dict(bytes=n * 6 * 6 * size, flops=n * 6 * flops)


# ---- the same outputs in FP64, plain torch -----------------------------------------

class _Fem:
    """Periodic trilinear elements with 2x2x2 Gauss points; fields are (R, N, 3), C is (N, 6, 6)."""

    def __init__(self, shape, h, C):
        self.shape, self.C = shape, C
        self.h = np.asarray(h, dtype=float)
        self.V = float(np.prod(self.h))
        g = 1 / math.sqrt(3)
        pts = [(a * g, b * g, c * g) for c in (-1, 1) for b in (-1, 1) for a in (-1, 1)]
        self.B = [torch.tensor(self._b(*p), dtype=torch.float64, device="cuda") for p in pts]
        self.B0 = torch.tensor(self._b(0, 0, 0), dtype=torch.float64, device="cuda")

    def _b(self, x, y, z):
        B = np.zeros((6, 24))
        for a in range(8):
            s = [1 if a >> d & 1 else -1 for d in range(3)]
            t = [1 + s[0] * x, 1 + s[1] * y, 1 + s[2] * z]
            d = [s[0] * t[1] * t[2] / (4 * self.h[0]), s[1] * t[0] * t[2] / (4 * self.h[1]),
                 s[2] * t[0] * t[1] / (4 * self.h[2])]
            for r, c, k in ((0, 0, 0), (1, 1, 1), (2, 2, 2), (3, 1, 2), (3, 2, 1), (4, 0, 2), (4, 2, 0), (5, 0, 1),
                            (5, 1, 0)):
                B[r, 3 * a + c] = d[k]
        return B

    def corners(self, u):
        g = u.reshape(-1, *self.shape, 3)
        return torch.cat([torch.roll(g, (-(a >> 2 & 1), -(a >> 1 & 1), -(a & 1)), (1, 2, 3)) for a in range(8)],
                         dim=-1).reshape(u.shape[0], -1, 24)

    def scatter(self, f):
        g = f.reshape(-1, *self.shape, 24)
        out = 0
        for a in range(8):
            out = out + torch.roll(g[..., 3 * a:3 * a + 3], (a >> 2 & 1, a >> 1 & 1, a & 1), (1, 2, 3))
        return out.reshape(f.shape[0], -1, 3)

    def stress(self, eps):
        return torch.matmul(self.C, eps.unsqueeze(-1)).squeeze(-1)

    def apply(self, u):
        out = torch.empty_like(u)
        for r in range(0, len(u), 6 if u.shape[1] < 300_000 else 1):
            part = slice(r, r + (6 if u.shape[1] < 300_000 else 1))
            e, f = self.corners(u[part]), 0
            for B in self.B:
                f = f + self.stress(e @ B.T) @ B * (self.V / 8)
            out[part] = self.scatter(f)
        return out

    def rhs(self, E):
        return torch.cat([self.scatter(-self.V * (self.stress(e.expand(1, self.C.shape[0], 6)) @ self.B0))
                          for e in E])

    def mean_stress(self, u, E):
        return torch.cat([(self.stress(self.corners(u[r:r + 1]) @ self.B0.T + E[r])).mean(1) for r in range(len(u))])

    def green(self, lam, mu):
        """M: the inverse symbol of the uniform isotropic medium; the constant mode goes to zero."""
        nz, ny, nx = self.shape
        ax = []
        for n, h, count, dim in ((nx, self.h[0], nx // 2 + 1, 2), (ny, self.h[1], ny, 1), (nz, self.h[2], nz, 0)):
            t = 2 * math.pi * torch.arange(count, dtype=torch.float64, device="cuda") / n
            s2 = torch.sin(t / 2) ** 2
            m = (2 + torch.cos(t)) / 3
            view = [1, 1, 1]
            view[dim] = count
            ax.append([v.reshape(view) for v in (m, 4 * s2 / (h * h * m), torch.sin(t) / (h * m),
                                                 4 * s2 * s2 / (3 * h * h * m * m))])
        D = ax[0][1] + ax[1][1] + ax[2][1]
        scale = 1 / (self.V * ax[0][0] * ax[1][0] * ax[2][0])
        scale[0, 0, 0] = 0
        D[0, 0, 0] = 1
        v = [a[2] for a in ax]
        i = [1 / (mu * D + (lam + mu) * a[3]) for a in ax]
        gamma = (lam + mu) / (1 + (lam + mu) * sum(a * a * b for a, b in zip(v, i)))

        def solve(r):
            out = torch.empty_like(r)
            for k in range(len(r)):
                q = torch.fft.rfftn(r[k].reshape(*self.shape, 3), dim=(0, 1, 2))
                w = [q[..., c] * i[c] for c in range(3)]
                dot = gamma * sum(v[c] * w[c] for c in range(3))
                z = torch.stack([scale * (w[c] - v[c] * i[c] * dot) for c in range(3)], dim=-1)
                out[k] = torch.fft.irfftn(z, s=self.shape, dim=(0, 1, 2)).reshape(-1, 3)
            return out
        return solve

    def solve(self, tol=1e-10, most=3000):
        """C_eff (6, 6) and the six fluctuation fields of the unit strains."""
        E = torch.eye(6, dtype=torch.float64, device="cuda")
        lam = float(self.C[:, 0, 1].mean())
        mu = float(self.C[:, 3, 3].mean())
        M = self.green(lam, mu)
        f = self.rhs(E)
        f = f - f.mean(1, keepdim=True)
        dot = lambda a, b: (a * b).sum((1, 2))[:, None, None]  # noqa: E731
        ff = dot(f, f).clamp_min(1e-300)
        u, r = torch.zeros_like(f), f.clone()
        z = M(r)
        p, rz = z.clone(), dot(r, z)
        for k in range(most):
            q = self.apply(p)
            pq = dot(p, q)
            a = torch.where(pq > 0, rz / pq.clamp_min(1e-300), torch.zeros_like(pq))
            u += a * p
            r -= a * q
            if k % 5 == 4 and float((dot(r, r) / ff).max()) < tol * tol:
                break
            z = M(r)
            new = dot(r, z)
            p = z + torch.where(rz > 0, new / rz.clamp_min(1e-300), torch.zeros_like(rz)) * p
            rz = new
        u = u - u.mean(1, keepdim=True)
        return self.mean_stress(u, E).T, u


def _material(spec):
    if spec["kind"] == "isotropic":
        return _isotropic(spec["E"], spec["nu"])
    return _orthotropic(spec) if spec["kind"] == "orthotropic" else np.asarray(spec["C"], dtype=float)


def _stiffness(labels, materials, orientation):
    """(N, 6, 6) stiffness of every voxel."""
    flat = torch.as_tensor(np.asarray(_host(labels)).reshape(-1).astype(np.int64), device="cuda")
    table = torch.tensor(np.stack([_material(materials[k]) for k in range(len(materials))]), device="cuda")
    C = table[flat]
    for k, spec in materials.items():
        if spec.get("frame") == "local":
            vox = torch.nonzero(flat == k).squeeze(1)
            a, b = (torch.as_tensor(orientation[x].reshape(-1, 3), device="cuda")[vox] for x in ("axis1", "axis2"))
            a = a / a.norm(dim=1, keepdim=True)
            b = b - (a * b).sum(1, keepdim=True) * a
            b = b / b.norm(dim=1, keepdim=True)
            T = _bond(torch.stack([a, b, torch.linalg.cross(a, b)], dim=2))
            C[vox] = T @ table[k] @ T.transpose(1, 2)
    return C


def _planes(v):
    return v.transpose(1, 2).contiguous()


def exact(case, seed):
    """What run() returns, in FP64 and without the package's kernels; None where that takes too long."""
    kind = case["kind"]
    if kind == "batch":
        out = []
        for phase, materials, domain in _batch_cells(case, seed):
            h = domain / np.array(phase.shape[::-1], dtype=float)
            out.append(_Fem(phase.shape, h, _stiffness(phase, materials, None)).solve()[0].cpu().numpy())
        return out
    shape = (case["nz"], case["ny"], case["nx"])
    n = case["nx"] * case["ny"] * case["nz"]
    if kind == "call":
        if n > 2_200_000:
            return None
        labels, materials, domain, orientation = _cell(case, seed)
        fem = _Fem(shape, domain / np.array(shape[::-1], dtype=float), _stiffness(labels, materials, orientation))
        return fem.solve()[0].cpu().numpy()
    if kind == "simp":
        rho = _density(case, seed).double().reshape(-1)
        C1 = torch.tensor(_isotropic(1.0, 0.3), device="cuda")
        E = 1e-3 + rho ** 3 * (70.0 - 1e-3)
        fem = _Fem(shape, [1.0 / s for s in shape[::-1]], E[:, None, None] * C1)
        CH, u = fem.solve(tol=1e-11)
        e, g = fem.corners(u), 0
        strain = torch.eye(6, dtype=torch.float64, device="cuda")[:, None, :]
        W = torch.zeros(6, 6, dtype=torch.float64, device="cuda")
        W[0, 0] = 1.0
        W[:3, :3] += 1.0 / 9.0
        for B in fem.B:
            eps = e @ B.T + strain
            g = g + (eps * torch.tensordot(W, eps @ C1, dims=1)).sum((0, 2)) * (fem.V / 8)
        grad = 3 * rho ** 2 * (70.0 - 1e-3) * g / (fem.V * n)
        return dict(C=CH.cpu(), grad=grad.reshape(shape))
    if kind == "precond":
        u = _randn((6, 3, n), seed, case["dtype"]).double()
        fem = _Fem(shape, (1.0 / case["nx"],) * 3, None)
        return _planes(fem.green(**_MEDIUM)(_planes(u)))
    cell = case if kind != "protocol" else dict(case, cell="grains", grains=20)
    labels, materials, domain, _ = _cell(cell, seed)
    fem = _Fem(shape, domain / np.array(shape[::-1], dtype=float), _stiffness(labels, materials, None))
    if kind == "protocol":
        u, r = (_randn((1, 3 * n), seed + k, "float64").reshape(1, n, 3) for k in (0, 1))
        return fem.apply(u).reshape(1, -1), fem.green(**_MEDIUM)(r).reshape(1, -1)
    if kind == "operator":
        return _planes(fem.apply(_planes(_randn((6, 3, n), seed, case["dtype"]).double())))
    u = _planes(_randn((6, 3, n), seed, "float64").mul_(1e-3))
    E = torch.eye(6, dtype=torch.float64, device="cuda")
    strain = torch.cat([fem.corners(u[k:k + 1]) @ fem.B0.T + E[k] for k in range(6)])
    stress = torch.cat([fem.stress(strain[k:k + 1]) for k in range(6)])
    return _planes(fem.rhs(E)), _planes(strain), _planes(stress), 0.5 * (strain * stress).sum(-1)
