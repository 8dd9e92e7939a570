"""Right-hand sides and element-centre fields against plain torch, at the edges of
the column march: axes of two nodes, one plane short of and past a chunk, ragged
planes, every output left out in turn."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

SHAPES = [(2, 2, 2), (3, 2, 5), (17, 16, 16), (16, 15, 33), (33, 3, 100), (5, 40, 41), (100, 96, 110)]
H = (1.0, 0.5, 1.5)


def _cell(shape, kind, scale=False):
    import torch
    from voxel_lmfem import materials as pm
    from voxel_lmfem.gpu import Cell
    rng = np.random.default_rng(5)
    rows = []
    for _ in range(3):
        a = rng.standard_normal((6, 6))
        rows.append(pm.pack21(a @ a.T + 6.0 * np.eye(6)))
    n = int(np.prod(shape))
    index = rng.integers(0, 3, n).astype(kind)
    s = rng.uniform(0.2, 1.0, n).astype(np.float32) if scale else None
    cell = Cell(pm.MaterialField(np.stack(rows), index, None, None, None), shape, H, scale=s)
    C = np.zeros((3, 6, 6))
    iu = np.triu_indices(6)
    for k in range(3):
        C[k][iu] = rows[k]
        C[k] = C[k] + np.triu(C[k], 1).T
    C = torch.from_numpy(C[index]).cuda()
    return cell, C if s is None else C * torch.from_numpy(s.astype(np.float64)).cuda()[:, None, None]


def _corner(v, shape, q, sign):
    """v at corner q of every element (sign -1) or element q around every node (+1)."""
    import torch
    ax, ay, az = q & 1, (q >> 1) & 1, q >> 2
    return torch.roll(v.reshape(*v.shape[:-1], *shape), (sign * az, sign * ay, sign * ax), (-3, -2, -1)).flatten(-3)


def _grad(q):
    return [(1 if q >> a & 1 else -1) * 0.25 / H[a] for a in range(3)]


@pytest.mark.parametrize("shape", SHAPES)
@pytest.mark.parametrize("kind,scale,nload", [(np.uint8, False, 6), (np.int32, True, 1)])
def test_center_fields(torch_gpu, shape, kind, scale, nload):
    torch = torch_gpu
    cell, C = _cell(shape, kind, scale)
    n = int(np.prod(shape))
    u = torch.randn(nload, 3, n, dtype=torch.float64, device="cuda", generator=torch.Generator("cuda").manual_seed(1))
    macro = np.random.default_rng(2).standard_normal((nload, 6))
    eps = torch.from_numpy(macro).cuda()[:, :, None].repeat(1, 1, n)
    for q in range(8):
        d, v = _grad(q), _corner(u, shape, q, -1)
        for i, pairs in enumerate([[(0, 0)], [(1, 1)], [(2, 2)], [(2, 1), (1, 2)], [(2, 0), (0, 2)], [(1, 0), (0, 1)]]):
            for a, c in pairs:
                eps[:, i] += d[a] * v[:, c]
    sig = torch.einsum("nij,rjn->rin", C, eps)
    got = cell.center_fields_planes(u, macro)
    want = (eps, sig, 0.5 * (eps * sig).sum(1))
    for g, w in zip(got, want):
        # Sums of some thirty terms in FP64.
        assert (g - w).abs().max() <= 64 * 2.3e-16 * w.abs().max() * 8
    cell.close()


@pytest.mark.parametrize("shape", SHAPES)
@pytest.mark.parametrize("kind,scale,nload", [(np.uint8, False, 6), (np.uint16, True, 1)])
def test_rhs(torch_gpu, shape, kind, scale, nload):
    torch = torch_gpu
    cell, C = _cell(shape, kind, scale)
    macro = np.random.default_rng(2).standard_normal((nload, 6))
    s = torch.einsum("nij,rj->rin", C, torch.from_numpy(macro).cuda())
    f = torch.zeros(nload, 3, s.shape[-1], dtype=torch.float64, device="cuda")
    voigt = [[0, 5, 4], [5, 1, 3], [4, 3, 2]]
    for q in range(8):
        d, v = _grad(q), _corner(s, shape, q, 1)
        for c in range(3):
            for a in range(3):
                f[:, c] -= H[0] * H[1] * H[2] * d[a] * v[:, voigt[c][a]]
    got = cell.rhs_planes(macro)
    top = s.abs().max() * H[0] * H[1] * H[2] * sum(abs(x) for x in _grad(7)) * 8
    assert (got - f).abs().max() <= 64 * 2.3e-16 * top
    cell.close()


# More than 1024 single planes of 256 columns: chunks of two planes and more, the last one short.
@pytest.mark.parametrize("shape", [(3, 190, 200), (7, 120, 101), (35, 150, 160)])
@pytest.mark.parametrize("kind,scale,nload", [(np.uint8, False, 6), (np.uint16, True, 3)])
def test_chunks_of_several_planes(torch_gpu, shape, kind, scale, nload):
    assert (shape[1] * shape[2] + 255) // 256 * nload * shape[0] > 1024 or nload == 3
    test_center_fields(torch_gpu, shape, kind, scale, nload)
    test_rhs(torch_gpu, shape, kind, scale, nload)
