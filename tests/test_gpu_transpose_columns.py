"""The exact transpose's kernel for circular orbits against the FP64 oracle
at the edges of its row windows, tiles and parts: relative L2 <= 1e-5,
pointwise <= 1e-4 * max|ref| (the parity bar)."""
import numpy as np
import pytest

import oracle
from conftest import assert_parity

pytestmark = pytest.mark.gpu

kk = pytest.importorskip("kernelkit")
from kernelkit import workloads  # noqa: E402
from kernelkit.geom.proj import Detector, ProjectionGeometry  # noqa: E402


def _dev(a):
    import torch
    return torch.from_numpy(np.ascontiguousarray(a, dtype=np.float32)).cuda()


def _orbit(angles, rows, cols, height, flip=False, shift=0.0, sod=150.0):
    """A circular orbit of magnification 1.5 with rows of ``height`` and
    columns of 1.2, rows upside down with ``flip``, the detector moved by
    ``shift`` along the axis."""
    det = Detector(rows=rows, cols=cols, pixel_height=height,
                   pixel_width=1.2)
    out = []
    for g in workloads.circular_geometry(angles, sod, sod / 2, rows, cols,
                                         1.2):
        v = np.asarray(g.v) * (-1 if flip else 1)
        d = np.asarray(g.detector_position) + shift * np.asarray(g.v)
        out.append(ProjectionGeometry(g.source_position, d, det, u=g.u, v=v))
    return out


def _check(pgs, shape, rows, cols, seed):
    vg = kk.resolve_volume_geometry(shape=shape, voxel_size=1.0)
    y = np.random.default_rng(seed).uniform(size=(len(pgs), rows, cols))
    got = kk.XrayTransform(pgs, vg).matched_T(_dev(y)).cpu().numpy()
    assert_parity(got, oracle.cone_fp_transpose(y, pgs, vg))


# rows per voxel: windows of 2, 3, 4 (coarse and fine), 5 ... 8, up to 12 and
# 16 rows, and longer ones
@pytest.mark.parametrize("flip", [False, True])
@pytest.mark.parametrize("fine", [0.5, 0.9, 1.05, 1.2, 1.55, 1.85, 2.15, 2.5,
                                  3.5, 4.2, 6.0, 40.0])
def test_row_windows(fine, flip, device):
    rows = int(24 * fine) + 2
    _check(_orbit(7, rows, 50, 1.5 / fine, flip), (23, 18, 21), rows, 50, 1)


# (shape, angles, rows, columns): lanes and b voxels past the volume, slices
# that fill no workgroup, several c tiles, one voxel, one pixel, one angle,
# more than 64 angles in a part, columns that leave the detector
@pytest.mark.parametrize("size", [((1, 1, 1), 1, 9, 9), ((9, 9, 1), 3, 1, 1),
                                  ((5, 17, 129), 5, 200, 40),
                                  ((18, 7, 260), 4, 300, 12),
                                  ((12, 16, 10), 530, 14, 22),
                                  ((33, 30, 40), 6, 30, 16)],
                         ids=str)
def test_tiles(size, device):
    shape, angles, rows, cols = size
    _check(_orbit(angles, rows, cols, 1.3, sod=4.0 * max(shape) + 20), shape,
           rows, cols, 2)


# detectors that see one end of the volume: windows far outside the detector
@pytest.mark.parametrize("shift", [-90.0, -30.0, 45.0, 400.0])
@pytest.mark.parametrize("flip", [False, True])
def test_detector_moved_along_the_axis(shift, flip, device):
    _check(_orbit(6, 40, 40, 1.0, flip, shift, sod=300.0), (20, 20, 140), 40,
           40, 3)


def test_rows_of_both_directions_and_tilted_angles(device):
    pgs = _orbit(10, 36, 44, 1.1)
    pgs = [p for k, p in enumerate(pgs) if k % 3] + \
        _orbit(5, 36, 44, 1.1, flip=True) + \
        [g for g in workloads.circular_geometry(
            4, 150.0, 75.0, 36, 44, 1.1, tilt_deg=2.0)]
    _check(pgs, (20, 24, 22), 36, 44, 4)


def test_two_and_four_parts_agree(device):
    """A volume large enough for two parts, and a slab of it (four parts):
    the same sums, split differently (float32: 1e-6 of the largest)."""
    pgs = _orbit(70, 60, 330, 1.1, sod=900.0)
    y = _dev(np.random.default_rng(5).uniform(size=(70, 60, 330)))
    whole = kk.resolve_volume_geometry(shape=(200, 200, 262), voxel_size=1.0)
    lo = np.array([-100.0, -100.0, -131.0])
    slab = kk.resolve_volume_geometry(
        shape=(40, 200, 262), extent_min=lo + [60, 0, 0],
        extent_max=lo + [100, 200, 262])
    a = kk.XrayTransform(pgs, whole).matched_T(y).cpu().numpy()
    b = kk.XrayTransform(pgs, slab).matched_T(y).cpu().numpy()
    assert np.abs(a[60:100] - b).max() <= 1e-6 * a.max()
