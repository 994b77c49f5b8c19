"""The exact transpose's walks at the edges of their windows and shares, against
the FP64 oracle: relative L2 <= 1e-5, pointwise <= 1e-4 * max|ref| (the parity
bar)."""
import numpy as np
import pytest

import oracle
from conftest import assert_parity

pytestmark = pytest.mark.gpu

kk = pytest.importorskip("kernelkit")
from kernelkit import workloads  # noqa: E402
from kernelkit.geom.proj import Detector, ProjectionGeometry  # noqa: E402


def _rolled_orbit(angles, rows, cols, height, roll, sod=150.0, width=1.2):
    """Orbit of magnification 1.5 about an axis ``roll`` degrees off z, the
    same way at all angles (rows then move one way along b)."""
    det = Detector(rows=rows, cols=cols, pixel_height=height,
                   pixel_width=width)
    c, s = np.cos(np.deg2rad(roll)), np.sin(np.deg2rad(roll))
    tilt = np.array([[1.0, 0.0, 0.0], [0.0, c, -s], [0.0, s, c]])
    out = []
    for k in range(angles):
        t = 2 * np.pi * k / angles + 0.09
        R = tilt @ np.array([[np.cos(t), -np.sin(t), 0.0],
                             [np.sin(t), np.cos(t), 0.0], [0.0, 0.0, 1.0]])
        out.append(ProjectionGeometry(
            R @ [-sod, 0.0, 0.0], R @ [0.5 * sod, 0.3, -0.4], det,
            u=R @ [0.0, 1.0, 0.0], v=R @ [0.0, 0.0, 1.0]))
    return out


# The unrolled walk where a column's rows are rounded up to the next unrolled
# length (9 -> 12, 13 -> 16) and their slope along b is at its limit.  Rows per
# voxel: windows of 9 and of 13 rows.
@pytest.mark.parametrize("sign", [1, -1])
@pytest.mark.parametrize("roll", [9.5, 10.0, 10.5, 10.9])
@pytest.mark.parametrize("fine", [1.75, 1.8, 1.85, 1.92, 2.7, 2.75, 2.8])
def test_padded_windows(fine, roll, sign, device):
    import torch
    rows = int(30 * fine) + 2
    pgs = _rolled_orbit(7, rows, 50, 1.5 / fine, sign * roll)
    vg = kk.resolve_volume_geometry(shape=(23, 18, 21), voxel_size=1.0)
    y = np.random.default_rng(1).uniform(size=(len(pgs), rows, 50))
    got = kk.XrayTransform(pgs, vg).matched_T(
        torch.from_numpy(y.astype(np.float32)).cuda()).cpu().numpy()
    assert_parity(got, oracle.cone_fp_transpose(y, pgs, vg))


# circular orbits of windows longer than the unrolled ones, all of the plan's
# angles or not (rows four at a time, or one by one), and around the rule's line
@pytest.mark.parametrize("tilted", [False, True])
@pytest.mark.parametrize("fine", [2.9, 3.2, 3.6, 5.0, 6.1, 11.0])
def test_long_windows_of_circular_orbits(fine, tilted, device):
    import torch
    rows = int(20 * fine) + 3
    pgs = []
    for kw in [{}] + [dict(tilt_deg=3.0)] * tilted:
        for g in workloads.circular_geometry(5, 120.0, 60.0, rows, 40, 1.1,
                                             **kw):
            det = Detector(rows=rows, cols=40, pixel_height=1.5 / fine,
                           pixel_width=1.1)
            pgs.append(ProjectionGeometry(g.source_position,
                                          g.detector_position, det, u=g.u,
                                          v=g.v))
    vg = kk.resolve_volume_geometry(shape=(20, 17, 19), voxel_size=1.0)
    y = np.random.default_rng(2).uniform(size=(len(pgs), rows, 40))
    got = kk.XrayTransform(pgs, vg).matched_T(
        torch.from_numpy(y.astype(np.float32)).cuda()).cpu().numpy()
    assert_parity(got, oracle.cone_fp_transpose(y, pgs, vg))


# angles of a launch per share or part: 1, 2, 4, 8 and 16 shares of general
# geometries, 1, 2 and 4 parts of circular orbits (volumes of few and of many
# workgroups)
@pytest.mark.parametrize("wobble", [0.5, 0.0])
@pytest.mark.parametrize("shape,angles", [
    ((20, 18, 17), 1), ((20, 18, 17), 2), ((20, 18, 17), 7),
    ((20, 18, 17), 24), ((20, 18, 17), 70), ((90, 80, 5), 9),
    ((90, 80, 5), 40), ((300, 280, 3), 4), ((300, 280, 3), 12),
    ((300, 280, 3), 30), ((300, 280, 3), 60)], ids=str)
def test_shares_of_the_angles(shape, angles, wobble, device):
    import torch
    m = max(shape)
    pgs = workloads.circular_geometry(angles, 3.0 * m, 1.5 * m, 12, 40,
                                      1.7 * m / 40, wobble_deg=wobble, seed=3)
    vg = kk.resolve_volume_geometry(shape=shape, voxel_size=1.0)
    y = np.random.default_rng(5).uniform(size=(angles, 12, 40))
    got = kk.XrayTransform(pgs, vg).matched_T(
        torch.from_numpy(y.astype(np.float32)).cuda()).cpu().numpy()
    assert_parity(got, oracle.cone_fp_transpose(y, pgs, vg))
