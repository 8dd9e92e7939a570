"""Stencil form of rows without normal-shear or shear-shear coupling: the same
bits as the general form (which an unused coupled row in the table selects),
and the oracle."""
import numpy as np
import pytest

from oracle import fem, materials as om
from voxel_lmfem import materials as pm

pytestmark = pytest.mark.gpu


def _fields(shape, seed, dtype):
    """(field that takes the orthotropic form, the same voxels with a coupled extra row, per-voxel 6x6)."""
    rng = np.random.default_rng(seed)
    rows = [pm.pack21(pm.isotropic_voigt(3.0, 0.35)), pm.pack21(pm.isotropic_voigt(70.0, 0.22)),
            pm.pack21(pm.orthotropic_voigt(135., 9., 11., .3, .28, .35, 5., 4., 3.5))]
    coupled = pm.pack21(np.eye(6) * 5 + 0.1)
    index = rng.integers(0, 3, size=int(np.prod(shape))).astype(dtype)
    plain = pm.MaterialField(np.stack(rows), index, None, None, None)
    general = pm.MaterialField(np.stack(rows + [coupled]), index, None, None, None)
    return plain, general, om.unpack21(np.stack(rows)[index.astype(np.int64)])


# Tile edges (32 x 14 / 6 / 8 / 4 nodes), remainders, the smallest grid; cubic and general voxels.
@pytest.mark.parametrize("shape,h", [((2, 2, 2), (1., 1., 1.)), ((5, 15, 33), (1., 1., 1.)), ((9, 14, 32), (.5, .7, .9)),
                                     ((7, 29, 40), (.3, 1.1, .8))])
@pytest.mark.parametrize("dtype", [np.uint8, np.uint16, np.int32])
def test_orthotropic_form_is_the_general_one(torch_gpu, shape, h, dtype):
    torch = torch_gpu
    from voxel_lmfem.gpu import Cell
    print(f"case ortho shape={shape} {np.dtype(dtype)}", flush=True)
    plain, general, full = _fields(shape, sum(shape), dtype)
    n = int(np.prod(shape))
    U = np.random.default_rng(1).normal(size=(2, n, 3))
    ref = np.stack([fem.MatrixFree(full, shape, np.array(h)).apply(u).T for u in U])
    a, b = Cell(plain, shape, h), Cell(general, shape, h)
    u = torch.tensor(np.ascontiguousarray(U.transpose(0, 2, 1)), device="cuda")
    for precision, tol, tiles in (("float64", 1e-13, (6, 8, 4)), ("float32", 2e-6, (14, 8, 6))):
        x = u.to(getattr(torch, precision))
        for ty in tiles:
            for cell in (a, b):
                cell.set_stencil_config(precision, ty, 3, 2)
            got, want = a.apply_planes(x), b.apply_planes(x)
            assert torch.equal(got, want)
            err = np.abs(got.double().cpu().numpy() - ref).max() / np.abs(ref).max()
            assert err < tol, (precision, ty, err)
    a.close()
    b.close()


@pytest.mark.parametrize("precision", ["mixed", "fp64"])
def test_solves_agree_bit_for_bit(torch_gpu, precision):
    from voxel_lmfem.gpu import Cell, Solver
    shape, h = (12, 17, 20), (1., 1., 1.2)
    print(f"case ortho solve {precision}", flush=True)
    plain, general, _ = _fields(shape, 4, np.uint8)
    out = []
    for field in (plain, general):
        cell = Cell(field, shape, h)
        solver = Solver(cell, 20.0, 12.0, mode=precision)
        out.append(solver.run(np.eye(6), return_fields=True))
        solver.close()
        cell.close()
    assert out[0]["iterations"] == out[1]["iterations"]
    assert np.array_equal(out[0]["CH"], out[1]["CH"])
    assert bool((out[0]["fields"] == out[1]["fields"]).all())
