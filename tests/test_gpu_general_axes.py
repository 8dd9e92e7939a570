"""The solver's forms on axes that take the general FFT passes: two in-register
factors, three, and a dense second factor; and mixed-mode right-hand sides far
from 1, whose FP32 recurrence is scaled by a power of two."""
import numpy as np
import pytest

from oracle import spectral
from voxel_lmfem import materials as pm

pytestmark = pytest.mark.gpu

# x last: two in-register factors; 37 and 34 dense; 147 three-step in FP64, 343 in both precisions.
SHAPES = [(21, 25, 18), (20, 37, 34), (6, 5, 147), (147, 6, 5), (5, 343, 4), (343, 4, 6)]


def rel(a, b):
    a, b = np.asarray(a, dtype=float), np.asarray(b, dtype=float)
    return float(np.linalg.norm(a - b) / np.linalg.norm(b))


def blocks(shape, seed, contrast=20.0, scale=1.0):
    """Two phases in random blocks of about three voxels."""
    rng = np.random.default_rng(seed)
    coarse = rng.random([s // 3 + 1 for s in shape]) < 0.4
    phase = coarse.repeat(3, 0).repeat(3, 1).repeat(3, 2)[:shape[0], :shape[1], :shape[2]].astype(np.int32)
    table = {0: dict(kind="isotropic", E=3.0 * scale, nu=0.3), 1: dict(kind="isotropic", E=3.0 * contrast * scale, nu=0.2)}
    return np.ascontiguousarray(phase), table, [float(s) for s in shape[::-1]]


def its(out):
    return [c["iterations"] for c in out["calls"]]


@pytest.mark.parametrize("precision", ["mixed", "fp64"])
@pytest.mark.parametrize("shape", SHAPES)
def test_solver_forms_agree(torch_gpu, monkeypatch, shape, precision):
    """Direction ring, fused residual update and spectral residual off in turn:
    iterations to one, C_eff to rounding."""
    from voxel_lmfem import homogenize
    args = blocks(shape, 2)
    print(f"case solver forms {shape} {precision}", flush=True)
    base = homogenize(*args, precision=precision)
    assert base["max_true_residual"] <= 1e-8
    for names in (("VXL_DIRECTION_RING",), ("VXL_SPECTRAL_RESIDUAL",), ("VXL_FUSED_UPDATE",),
                  ("VXL_DIRECTION_RING", "VXL_SPECTRAL_RESIDUAL")):
        with monkeypatch.context() as m:
            for name in names:
                m.setenv(name, "0")
            out = homogenize(*args, precision=precision)
        assert max(abs(a - b) for a, b in zip(its(out), its(base))) <= 1, names
        assert out["max_true_residual"] <= 1e-8 and rel(out["CH"], base["CH"]) < 1e-8, names


@pytest.mark.parametrize("mode", ["mixed", "fp64"])
@pytest.mark.parametrize("shape", SHAPES)
def test_stacked_cells_keep_their_media(torch_gpu, shape, mode):
    """Each stacked cell is preconditioned by its own medium: the iterations and
    stiffness of the single solves."""
    from voxel_lmfem.gpu import Cell, Solver
    from voxel_lmfem.reference_medium import select
    print(f"case stacked {shape} {mode}", flush=True)
    fields, media = [], []
    for k, (contrast, scale) in enumerate(((5.0, 1.0), (40.0, 1.0), (10.0, 30.0))):
        phase, table, _ = blocks(shape, k, contrast, scale)
        fields.append(pm.build_field(phase, table))
        media.append(select(fields[-1], phase, table)[:2])
    single = []
    for field, (lam, mu) in zip(fields, media):
        cell = Cell(field, shape, (1.0, 1.0, 1.0))
        solver = Solver(cell, lam, mu, mode=mode)
        single.append(solver.run())
        solver.close()
        cell.close()
    cell = Cell.stack(fields, shape, (1.0, 1.0, 1.0))
    solver = Solver(cell, [m[0] for m in media], [m[1] for m in media], mode=mode)
    out = solver.run()
    solver.close()
    cell.close()
    for g, one in enumerate(single):
        cols = slice(6 * g, 6 * g + 6)
        assert rel(np.asarray(out["CH"])[:, cols], one["CH"]) < 1e-8
        assert max(abs(int(a) - int(b)) for a, b in zip(out["iterations"][cols], one["iterations"])) <= 1
        assert max(out["true_residuals"][cols]) <= 1e-8


@pytest.mark.parametrize("shape", [(37, 4, 3), (118, 3, 4), (100, 4, 3), (147, 3, 4), (343, 2, 3), (3, 37, 100),
                                   (4, 3, 118)])
def test_hg_green_on_general_axes(torch_gpu, shape):
    """The C3D8R-HG symbol in the z pass with a dense second factor, with 32 and
    fewer columns a workgroup, and in three steps."""
    torch = torch_gpu
    from voxel_lmfem.gpu import Cell, Preconditioner
    print(f"case hg green general shape={shape}", flush=True)
    h = np.array([0.7, 1.1, 0.9])
    field = pm.build_field(np.zeros(shape, dtype=np.int32), {0: dict(kind="isotropic", E=1.0, nu=0.3)})
    cell = Cell(field, shape, h, element="c3d8r_hg", hourglass_coefficient=0.2)
    lam, mu, n = 2.5, 1.3, int(np.prod(shape))
    R = np.random.default_rng(6).normal(size=(2, n, 3))
    R -= R.mean(axis=1, keepdims=True)
    want = np.stack([spectral.green_hg_dense(r, shape, h, lam, mu, 0.2).T for r in R])
    r = torch.tensor(np.stack([np.ascontiguousarray(x.T) for x in R]), device="cuda")
    for precision, tol in (("float64", 1e-11), ("float32", 5e-6)):
        pc = Preconditioner(cell, lam, mu, precision=precision, nrhs_max=2)
        z = pc.apply_planes(r.to(pc.dtype)).double().cpu().numpy()
        err = np.abs(z - want).max() / np.abs(want).max()
        print(f"  {precision} err {err:.2e}", flush=True)
        assert err < tol
        pc.close()
    cell.close()


@pytest.mark.parametrize("ring", ["1", "0"])
@pytest.mark.parametrize("power", [40, -60])
@pytest.mark.parametrize("shape", [(16, 16, 16), (21, 25, 18)])
def test_moduli_far_from_one(torch_gpu, monkeypatch, shape, power, ring):
    """Moduli times 2^power (pascals instead of gigapascals and beyond): the
    right-hand sides are scaled by an exact power of two, so the solve takes the
    same steps and C_eff is the same but for that power."""
    from voxel_lmfem import homogenize
    monkeypatch.setenv("VXL_DIRECTION_RING", ring)
    print(f"case moduli 2^{power} {shape} ring={ring}", flush=True)
    base = homogenize(*blocks(shape, 3), precision="mixed")
    out = homogenize(*blocks(shape, 3, scale=2.0 ** power), precision="mixed")
    assert its(out) == its(base) and out["max_true_residual"] <= 1e-8
    assert rel(np.asarray(out["CH"]) * 2.0 ** -power, base["CH"]) < 1e-12


@pytest.mark.parametrize("ring", ["1", "0"])
@pytest.mark.parametrize("shape", [(16, 16, 16), (21, 25, 18)])
def test_some_loads_far_from_one(torch_gpu, monkeypatch, shape, ring):
    """Only some right-hand sides are scaled: each load's stress is that of the
    unit load times its size, and so is its displacement field."""
    from voxel_lmfem.gpu import Cell, Solver
    from voxel_lmfem.reference_medium import select
    monkeypatch.setenv("VXL_DIRECTION_RING", ring)
    print(f"case mixed load sizes {shape} ring={ring}", flush=True)
    phase, table, _ = blocks(shape, 4)
    field = pm.build_field(phase, table)
    lam, mu = select(field, phase, table)[:2]
    cell = Cell(field, shape, (1.0, 1.0, 1.0))
    solver = Solver(cell, lam, mu, mode="mixed")
    size = 2.0 ** np.array([0, 50, 0, -70, 0, 30])
    unit = solver.run(np.eye(6) * 2.0, return_fields=True)   # not the six unit strains: the same stress path
    u = unit["fields"].clone()
    out = solver.run(np.eye(6) * 2.0 * size[:, None], return_fields=True)
    v = out["fields"]
    assert list(out["iterations"]) == list(unit["iterations"])
    for k in range(6):
        assert rel(np.asarray(out["CH"])[:, k] / size[k], np.asarray(unit["CH"])[:, k]) < 1e-12
        assert float((v[k] / size[k] - u[k]).abs().max()) <= 1e-12 * float(u[k].abs().max())
    solver.close()
    cell.close()
