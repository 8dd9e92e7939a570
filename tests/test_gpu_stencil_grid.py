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


@pytest.mark.parametrize("precision", ["float32", "float64"])
@pytest.mark.parametrize("nrhs", [1, 6])
def test_chunk_depth_is_a_lower_bound(torch_gpu, precision, nrhs):
    """Depths 2 to 64 bound the planes per chunk from below (8 among them), 0 is
    the automatic depth of a new cell, and the kernel form names the table."""
    from voxel_lmfem import materials as pm
    from voxel_lmfem.gpu import Cell
    general = pm.isotropic_voigt(7.0, 0.3)
    general[0, 3] = general[3, 0] = 0.4
    rows = np.stack([pm.pack21(pm.isotropic_voigt(3.0, 0.35)), pm.pack21(general)])
    shape = (40, 20, 24)
    index = np.zeros(int(np.prod(shape)), dtype=np.uint8)
    for count, h, form in ((1, (1.0, 1.0, 1.0), "ortho+cubic"), (1, (1.0, 1.0, 1.5), "ortho"),
                           (2, (1.0, 1.0, 1.0), "cubic"), (2, (1.0, 1.0, 1.5), "")):
        cell = Cell(pm.MaterialField(rows[:count], index, None, None, None), shape, h)
        tile, schedule, zmin = cell.stencil_config(precision)
        assert zmin == 0
        _, automatic, got = cell.stencil_launch(precision, nrhs)
        assert got == form and 2 <= automatic < 8   # a small grid: more chunks than depth 8 allows
        for bound in (2, 4, 8, 16, 64):
            cell.set_stencil_config(precision, tile, schedule, bound)
            depth = cell.stencil_launch(precision, nrhs)[1]
            assert min(bound, shape[0]) <= depth <= shape[0]
            assert bound != 2 or depth == automatic
        cell.set_stencil_config(precision, tile, schedule, 0)
        assert cell.stencil_launch(precision, nrhs)[1] == automatic
        for refused in (1, -1, 65):
            with pytest.raises(ValueError):
                cell.set_stencil_config(precision, tile, schedule, refused)
        cell.close()


@pytest.mark.parametrize("shape,tile", [((32, 32, 32), (32, 6)), ((72, 16, 84), (32, 6)), ((2, 3, 2), (32, 6)),
                                        ((9, 13, 33), (32, 6)), ((64, 64, 64), (16, 14)), ((17, 56, 48), (16, 14))])
def test_default_fp64_tile_by_grid(torch_gpu, shape, tile):
    """FP64's option 6 is 32 x 6 or 16 x 14 by the grid; both give the sums of the
    other options (1e-13 as for every configuration), in the general and the
    orthotropic form and under the other schedules."""
    torch = torch_gpu
    from voxel_lmfem import materials as pm
    from voxel_lmfem.gpu import Cell
    rng = np.random.default_rng(5)
    general = pm.isotropic_voigt(7.0, 0.3)
    general[0, 3] = general[3, 0] = 0.4
    rows = np.stack([pm.pack21(pm.isotropic_voigt(3.0, 0.35)), pm.pack21(general)])
    n = int(np.prod(shape))
    index = (rng.random(n) < 0.4).astype(np.uint8)
    u = torch.from_numpy(rng.standard_normal((6, 3, n))).to("cuda")
    for count in (1, 2):
        cell = Cell(pm.MaterialField(rows[:count], index * (count - 1), None, None, None), shape, (1.0, 1.0, 1.5))
        assert cell.stencil_launch("float64", 6)[0] == tile
        cell.set_stencil_config("float64", 8, 3, 0)
        want = cell.apply_planes(u).clone()
        for schedule in (3, 2, 1):
            cell.set_stencil_config("float64", 6, schedule, 0)
            got = cell.apply_planes(u)
            assert float((got - want).abs().max()) <= 1e-13 * float(want.abs().max()), (count, schedule)
        cell.close()
