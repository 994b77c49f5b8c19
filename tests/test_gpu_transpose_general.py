"""The exact transpose's kernel for general geometries (tilted detectors,
wobbling orbits) against the FP64 oracle at the edges of its row windows,
tiles and shares: relative L2 <= 1e-5, pointwise <= 1e-4 * max|ref| (the
parity bar)."""
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


def _about(axis, deg):
    a = np.deg2rad(deg)
    i, j = [(1, 2), (2, 0), (0, 1)][axis]
    R = np.eye(3)
    R[i, i] = R[j, j] = np.cos(a)
    R[i, j], R[j, i] = -np.sin(a), np.sin(a)
    return R


def _orbit(angles, rows, cols, height, roll=0.0, pitch=0.0, sod=150.0,
           width=1.2):
    """Orbit of magnification 1.5 about a rotation axis off the z axis by
    ``roll`` and ``pitch`` degrees, another way at every second angle."""
    det = Detector(rows=rows, cols=cols, pixel_height=height,
                   pixel_width=width)
    out = []
    for k in range(angles):
        s = 1 if k % 2 else -1
        R = (_about(1, s * pitch) @ _about(0, s * roll)
             @ _about(2, 360.0 * k / angles + 5.0))
        out.append(ProjectionGeometry(
            R @ [-sod, 0.0, 0.0], R @ [0.5 * sod, 0.3, -0.4], det,
            u=R @ [0.0, 1.0, 0.0], v=R @ [0.0, 0.0, 1.0]))
    return out


def _check(pgs, shape, rows, cols, seed):
    vg = kk.resolve_volume_geometry(shape=shape, voxel_size=1.0)
    y = np.random.default_rng(seed).uniform(size=(len(pgs), rows, cols))
    got = kk.XrayTransform(pgs, vg).matched_T(_dev(y)).cpu().numpy()
    assert_parity(got, oracle.cone_fp_transpose(y, pgs, vg))


# rows per voxel: windows of 2 ... 8, up to 12 and 16 rows, and longer ones;
# slopes along b whose windows stay within a voxel, and steeper ones
@pytest.mark.parametrize("roll", [0.5, 4.0, 14.0, 35.0])
@pytest.mark.parametrize("fine", [0.3, 0.6, 0.9, 1.2, 1.5, 1.8, 2.2, 3.2, 4.4,
                                  9.0])
def test_row_windows(fine, roll, device):
    rows = int(30 * fine) + 2
    _check(_orbit(7, rows, 50, 1.5 / fine, roll, 0.7), (23, 18, 21), rows, 50,
           1)


# (shape, angles, rows, columns): lanes and b voxels past the volume, several
# c tiles, one voxel, one pixel, fewer angles than shares, and volumes whose
# angles go to 16, 8 and 4 shares
@pytest.mark.parametrize("size", [((1, 1, 1), 1, 9, 9), ((9, 9, 1), 3, 1, 1),
                                  ((5, 17, 129), 5, 200, 40),
                                  ((18, 7, 260), 4, 300, 12),
                                  ((12, 16, 10), 130, 14, 22),
                                  ((90, 136, 3), 21, 6, 90),
                                  ((512, 500, 2), 5, 5, 60)])
def test_sizes(size, device):
    shape, angles, rows, cols = size
    _check(_orbit(angles, rows, cols, 1.3, 1.0, -0.8,
                  sod=3.0 * max(30, max(shape[:2])),
                  width=1.2 * max(1.0, max(shape[:2]) / cols)),
           shape, rows, cols, 2)


# sources close to the volume: the magnification differs along a window
@pytest.mark.parametrize("sod", [14.0, 20.0, 40.0])
def test_close_source(sod, device):
    _check(_orbit(6, 40, 44, 1.0, 3.0, 6.0, sod=sod), (15, 14, 13), 40, 44, 3)
