"""The stencil's launch grid (tiles and z chunks) never shows in its results: the
depth the launch chooses by itself gives the bits of one chunk per column."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape", [(2, 3, 2), (3, 14, 33), (7, 15, 17), (21, 25, 18), (64, 30, 31), (37, 92, 70),
                                   (111, 94, 118)])
@pytest.mark.parametrize("nrhs", [1, 6])
def test_chunk_rule_is_bitwise_neutral(torch_gpu, shape, nrhs):
    torch = torch_gpu
    from voxel_lmfem import materials as pm
    from voxel_lmfem.gpu import Cell
    rng = np.random.default_rng(3)
    general = pm.isotropic_voigt(7.0, 0.3)
    general[0, 3] = general[3, 0] = 0.4
    rows = np.stack([pm.pack21(pm.isotropic_voigt(3.0, 0.35)), pm.pack21(general)])
    n = int(np.prod(shape))
    index = (rng.random(n) < 0.4).astype(np.uint8)
    for count in (1, 2):  # the orthotropic and the general form
        cell = Cell(pm.MaterialField(rows[:count], index * (count - 1), None, None, None), shape, (1.0, 1.0, 1.5))
        for precision in ("float32", "float64"):
            u = torch.from_numpy(rng.standard_normal((nrhs, 3, n))).to("cuda", getattr(torch, precision))
            tile, schedule, depth = cell.stencil_config(precision)
            got = cell.apply_planes(u).clone()
            cell.set_stencil_config(precision, tile, schedule, 64)
            assert torch.equal(got, cell.apply_planes(u)), (count, precision)
            cell.set_stencil_config(precision, tile, schedule, depth)
        cell.close()
