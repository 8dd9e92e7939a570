"""The library's threaded host passes against NumPy (no GPU)."""
import numpy as np
import pytest

from voxel_lmfem import _native, inputs, materials as pm
from voxel_lmfem.solver import _pack_labels


@pytest.mark.parametrize("dtype", [np.uint8, np.int8, np.uint16, np.int16, np.uint32, np.int32, np.int64])
@pytest.mark.parametrize("size", [1, 7, (1 << 18) + 3])
def test_label_passes_match_numpy(dtype, size):
    rng = np.random.default_rng(size)
    info = np.iinfo(dtype)
    lo, hi = max(info.min, -90), min(info.max, 165)
    flat = np.repeat(rng.integers(lo, hi + 1, size=size // 3 + 1), 3)[:size].astype(dtype)
    flat[-1] = hi
    assert _native.host_labels(flat) is not None
    phase = flat.reshape(1, 1, -1)
    got = inputs.used_labels(phase)
    want = np.unique(flat)
    assert got.dtype == want.dtype and np.array_equal(got, want)
    for label in (int(flat[0]), hi, 300):
        assert np.array_equal(pm.voxels_with_label(flat, label), np.flatnonzero(flat == label))
    packed = _pack_labels(phase, {int(v): None for v in want})
    if size >= (1 << 18) and info.bits > 8:
        values, base = packed
        assert values.dtype == np.uint8 and np.array_equal(values.astype(np.int64) + base, phase)
    else:
        assert packed is None


def test_wide_labels_pack_to_16_bits_and_stay_out_beyond():
    flat = np.arange(1 << 18, dtype=np.int64) % 60000 - 5
    table = {int(v): None for v in range(-5, 59995)}
    values, base = _pack_labels(flat.reshape(64, 64, 64), table)
    assert values.dtype == np.int16 and base == -5
    assert np.array_equal(values.view(np.uint16).astype(np.int64) + base, flat.reshape(64, 64, 64))
    assert _pack_labels(flat.reshape(64, 64, 64), {0: None, 1 << 20: None}) is None


@pytest.mark.parametrize("labels", [np.array([5, 1 << 40], dtype=np.int64), np.array([3, 2 ** 63], dtype=np.uint64),
                                    np.arange(12, dtype=np.int32)[::2], np.arange(6, dtype=">i4")])
def test_labels_outside_the_native_passes(labels):
    got = inputs.used_labels(labels.reshape(1, 1, -1))
    assert np.array_equal(got, np.unique(labels))


@pytest.mark.parametrize("plant", [None, ("axis1", 40, np.nan), ("axis2", 41, np.inf), ("axis1", 17, 0.0),
                                   ("axis2", 60, "line")])
@pytest.mark.parametrize("second", [None, ("axis1", 90, np.nan), ("axis2", 45, 0.0)])
def test_axis_checks_match_the_numpy_pieces(plant, second):
    rng = np.random.default_rng(3)
    shape = (4, 5, 6)
    ori = {k: rng.normal(size=shape + (3,)) for k in ("axis1", "axis2")}
    for p in (plant, second):
        if p is not None:
            row = ori[p[0]].reshape(-1, 3)[p[1]]
            row[:] = 2.5 * ori["axis1"].reshape(-1, 3)[p[1]] if p[2] == "line" else p[2]
    sels = [np.arange(10, 70), np.zeros(0, dtype=np.int64), np.arange(70, 120, 2)]

    def outcome(native):
        try:
            src = ori if native else {k: np.asfortranarray(v) for k, v in ori.items()}  # strided: the NumPy pieces
            return pm.check_frames(src, shape, sels, chunk=16, workers=3, keep=True)
        except ValueError as exc:
            return str(exc)
    got, want = outcome(True), outcome(False)
    if isinstance(want, str):
        assert got == want
    else:
        assert all(np.array_equal(a, b) for a, b in zip(got, want))


@pytest.mark.parametrize("dtype,labels", [(np.uint8, 2), (np.uint8, 251), (np.int16, 300), (np.int32, 16384),
                                          (np.int32, 16385), (np.int64, 100000)])
@pytest.mark.parametrize("size", [1, 31, 32, 33, (1 << 18) - 1, (1 << 18), (1 << 19) + 5])
def test_labels_in_no_order(dtype, labels, size):
    """Random labels: narrow ranges (a table per piece) and wide ones (a shared
    table), one piece and several, groups of 32 with and without a match."""
    rng = np.random.default_rng(size + labels)
    flat = rng.integers(0, labels, size).astype(dtype)
    if size > 2:
        flat[[0, -1]] = 0, labels - 1
    assert np.array_equal(inputs.used_labels(flat.reshape(1, 1, -1)), np.unique(flat))
    for label in {int(flat[0]), int(flat[-1]), labels // 2, labels}:
        assert np.array_equal(pm.voxels_with_label(flat, label), np.flatnonzero(flat == label))


def _misaligned(a):
    """The same array one byte past its item alignment."""
    out = np.ndarray(a.shape, a.dtype, bytearray(a.nbytes + a.itemsize), offset=1)
    out[...] = a
    assert out.flags.c_contiguous and not out.flags.aligned
    return out


@pytest.mark.parametrize("dtype", [np.uint16, np.int32, np.int64])
def test_misaligned_labels_take_the_numpy_route(dtype):
    phase = _misaligned(np.random.default_rng(1).integers(0, 40, (1, 512, 520)).astype(dtype))
    assert _native.host_labels(phase.reshape(-1)) is None
    assert np.array_equal(inputs.used_labels(phase), np.unique(phase))
    assert np.array_equal(pm.voxels_with_label(phase.reshape(-1), 7), np.flatnonzero(phase == 7))
    assert _pack_labels(phase, {v: None for v in range(40)}) is None


def test_misaligned_axes_take_the_numpy_route():
    rng = np.random.default_rng(3)
    shape = (4, 5, 6)
    ori = {k: _misaligned(rng.normal(size=shape + (3,))) for k in ("axis1", "axis2")}
    kept = tuple(np.empty((60, 3)) for _ in range(2))
    sels = [np.arange(10, 70)]
    assert not pm._native_axes((ori["axis1"], ori["axis2"]), shape, sels, 16, 2, kept)
    got = pm.check_frames(ori, shape, sels, chunk=16, workers=2, keep=True)
    assert all(np.array_equal(g, ori[k].reshape(-1, 3)[10:70]) for g, k in zip(got, ("axis1", "axis2")))


@pytest.mark.parametrize("label", [2 ** 64 + 1, -2 ** 64 + 1, 2 ** 63])
def test_labels_past_64_bits_match_nothing(label):
    """They must not wrap to a label that is there."""
    flat = np.array([1, 2, 1, -2 ** 31], dtype=np.int32)
    try:
        got = pm.voxels_with_label(flat, label)
    except OverflowError:   # what NumPy's comparison raises in some versions
        return
    assert len(got) == 0
