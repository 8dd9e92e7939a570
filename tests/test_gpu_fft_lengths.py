"""Preconditioner on axes of any length against the oracle: in-register pairs,
dense second factors (prime factors above 13), primes, and the longest axes,
on each axis in turn."""
import numpy as np
import pytest

from oracle import spectral
from voxel_lmfem import materials as pm

pytestmark = pytest.mark.gpu

# 2 to 25: one or two small factors; 17, 19, 34 = 2*17, 37, 59*2, 61, 101, 127, 251: dense factors (odd and even);
# 100, 125, 150, 169, 225: in-register pairs; 64, 96, 256: lengths of the four-step kernels, run through the general
# passes; 323 = 17*19, 343 = 7*49, 512.
LENGTHS = [2, 3, 5, 7, 9, 11, 13, 14, 17, 18, 19, 20, 21, 22, 25, 34, 37, 61, 64, 96, 100, 101, 118, 125, 127, 150, 169,
           225, 251, 256, 323, 343, 512]


def _check(torch, shape, h, nrhs, precisions=(("float64", 1e-11), ("float32", 5e-6))):
    from voxel_lmfem.gpu import Cell, Preconditioner
    print(f"case lengths shape={shape}", flush=True)
    C = {0: dict(kind="isotropic", E=1.0, nu=0.3)}
    field = pm.build_field(np.zeros(shape, dtype=np.int32), C)
    cell = Cell(field, shape, h)
    lam, mu = 2.5, 1.3
    n = int(np.prod(shape))
    R = np.random.default_rng(n).normal(size=(nrhs, n, 3))
    R -= R.mean(axis=1, keepdims=True)
    ref = np.stack([spectral.green_apply(r, shape, h, lam, mu).T for r in R])
    r = torch.tensor(np.ascontiguousarray(R.transpose(0, 2, 1)), device="cuda")
    for precision, tol in precisions:
        pc = Preconditioner(cell, lam, mu, precision=precision, nrhs_max=nrhs)
        z = pc.apply_planes(r.to(pc.dtype)).double().cpu().numpy()
        err = np.abs(z - ref).max() / np.abs(ref).max()
        print(f"  {precision} err {err:.2e}", flush=True)
        assert err < tol
        pc.close()
    cell.close()


@pytest.mark.parametrize("n", LENGTHS)
def test_every_axis_length(torch_gpu, n, monkeypatch):
    monkeypatch.setenv("VXL_FFT_FOURSTEP", "0")
    monkeypatch.setenv("VXL_FFT_XFOURSTEP", "0")
    h = np.array([0.7, 1.1, 0.9])
    for shape in ((3, 5, n), (3, n, 5), (n, 5, 3)):
        _check(torch_gpu, shape, h, 2)


# Many columns per workgroup on all three axes at once, with partly filled last workgroups.
@pytest.mark.parametrize("shape", [(21, 25, 18), (33, 34, 35), (37, 50, 47), (30, 118, 26)])
def test_ragged_grids(torch_gpu, shape):
    _check(torch_gpu, shape, np.array([1.0, 1.0, 1.5]), 2)


# The longest axes the passes take (more than 64 KB of LDS in one workgroup).
@pytest.mark.parametrize("shape,precision,tol", [((2, 2, 1365), "float32", 2e-5), ((1365, 2, 2), "float32", 2e-5),
                                                 ((2, 4096, 2), "float32", 2e-5), ((2, 2, 682), "float64", 1e-10),
                                                 ((682, 2, 2), "float64", 1e-10), ((2, 2048, 2), "float64", 1e-10)])
def test_longest_axes(torch_gpu, shape, precision, tol):
    _check(torch_gpu, shape, np.array([1.0, 1.0, 1.0]), 1, ((precision, tol),))


# Lengths whose factors are all small but no in-register pair: three steps (FP64, or both precisions), with 64, 32, 16
# and fewer columns a workgroup, odd row counts and every middle factor; the last ones lie past 682 in FP64.
@pytest.mark.parametrize("n", [27, 44, 63, 99, 147, 175, 189, 200, 216, 243, 250, 264, 270, 288, 336, 375, 392, 448, 486,
                               500, 539, 605, 625, 675, 700, 720, 729, 1000, 1014, 1280, 1331])
def test_three_step_lengths(torch_gpu, n):
    h = np.array([0.7, 1.1, 0.9])
    tols = (("float64", 1e-11), ("float32", 5e-6)) if n <= 512 else (("float64", 1e-10), ("float32", 2e-5))
    for shape in ((3, 5, n), (3, n, 5), (n, 5, 3)):
        _check(torch_gpu, shape, h, 2, tols)


@pytest.mark.parametrize("shape", [(16, 16, 16), (9, 10, 14), (37, 6, 34)])
def test_denominators_past_the_largest_double(torch_gpu, shape):
    """Entries of the C3D8R-HG symbol beyond 1.8e308 have reciprocal 0, not NaN: with
    mu = 1e308 and h = 0.1 most wavevectors have one, and what is left is below
    1e-300.  (The FI symbol subtracts two such terms, so that it has none.)"""
    torch = torch_gpu
    from voxel_lmfem.gpu import Cell, Preconditioner
    field = pm.build_field(np.zeros(shape, dtype=np.int32), {0: dict(kind="isotropic", E=1.0, nu=0.3)})
    cell = Cell(field, shape, np.full(3, 0.1), element="c3d8r_hg")
    pc = Preconditioner(cell, 0.0, 1e308, precision="float64", nrhs_max=1)
    r = torch.from_numpy(np.random.default_rng(4).normal(size=(1, 3, int(np.prod(shape))))).to("cuda")
    z = pc.apply_planes(r)
    assert bool(torch.isfinite(z).all()) and float(z.abs().max()) < 1e-300
    pc.close()
    cell.close()
