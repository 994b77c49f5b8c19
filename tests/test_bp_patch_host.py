"""Host side of the backprojector's patch kernel: the bounds on the detector
patches of its tiles."""
import numpy as np
import pytest

kk = pytest.importorskip("kernelkit")
from kernelkit import _native, workloads  # noqa: E402
from kernelkit.kernels.cone_bp import VoxelDrivenConeBP  # noqa: E402


def _extent(pgs, vg):
    p = np.ascontiguousarray(VoxelDrivenConeBP.geoms2params(pgs, vg))
    out = np.zeros(2)
    _native.check(_native.lib().kk_bp_patch_extent(
        _native.f64_ptr(p), len(pgs), _native.i32(vg.shape),
        _native.f64_ptr(out)))
    return p.reshape(-1, 3, 4), out


@pytest.mark.parametrize("shape,sod,odd,pixel,centre", [
    ((64, 64, 64), 150.0, 75.0, 1.0, (0, 0, 0)),
    ((50, 33, 90), 60.0, 200.0, 2.5, (0, 0, 0)),
    ((17, 80, 7), 60.0, 30.0, 3.0, (4.0, -3.0, 9.0)),
])
@pytest.mark.parametrize("pert", [{}, {"wobble_deg": 1.0, "drift_px": 3.0},
                                  {"wobble_deg": 20.0, "tilt_deg": 15.0}])
def test_extent_covers_every_tile(shape, sod, odd, pixel, centre, pert):
    """The taps of every 16 x 16 x 16 tile (z beyond the volume to the end of
    its run) span no more columns and rows than the bounds."""
    pgs = workloads.circular_geometry(37, sod, odd, 40, 40, pixel, **pert)
    lo = np.array(centre) - 0.5 * np.array(shape)
    vg = kk.resolve_volume_geometry(shape=shape, voxel_size=1.0,
                                    extent_min=tuple(lo),
                                    extent_max=tuple(lo + np.array(shape)))
    P, out = _extent(pgs, vg)
    worst = np.zeros(2)
    tiles = [(x, min(x + 15, shape[0] - 1), y, min(y + 15, shape[1] - 1), z,
              z + 15) for x in range(0, shape[0], 16)
             for y in range(0, shape[1], 16) for z in range(0, shape[2], 16)]
    T = np.array(tiles, dtype=float)
    T -= 0.5 * np.repeat(shape, 2) - 0.5
    for nu, nv, de in P:
        lims = []
        for num in (nu, nv):
            c = []
            for e in range(8):
                X = T[:, [e & 1, 2 + (e >> 1 & 1), 4 + (e >> 2)]]
                c.append((num[3] + X @ num[:3]) / (de[3] + X @ de[:3]) + 0.5)
            c = np.array(c)
            lims.append(np.floor(c.max(0)) + 2 - np.floor(c.min(0)))
        worst = np.maximum(worst, [lims[0].max(), lims[1].max()])
    assert (worst <= out).all(), (worst, out)


def test_extent_refuses_other_geometries():
    vg = kk.resolve_volume_geometry(shape=(32, 32, 32), voxel_size=1.0)
    pgs = workloads.circular_geometry(8, 100.0, 50.0, 40, 40, 1.0,
                                      tilt_deg=1.0)
    assert _extent(pgs, vg)[1][0] < 0
    # the source's plane crosses the volume
    for kw in ({}, dict(wobble_deg=1.0)):
        pgs = workloads.circular_geometry(8, 10.0, 50.0, 40, 40, 1.0, **kw)
        assert _extent(pgs, vg)[1][0] < 0


@pytest.mark.parametrize("n", [0, 1, 7])
def test_cross_products_are_numpys_to_the_bit(n):
    from kernelkit.kernels.cone_bp import _cross
    r = np.random.default_rng(n)
    a, b = r.normal(size=(n, 3)), r.normal(size=(3, n)).T
    assert np.array_equal(_cross(a, b), np.cross(a, b))


def test_isotropic_voxels_of_equal_close_and_unequal_sizes():
    for step, expected in ((0.0, True), (2e-6, True), (1e-3, False)):
        vg = kk.VolumeGeometry((4, 4, 4), (1.0, 1.0, 1.0 + step),
                               (-2.0, -2.0, -2.0), (2.0, 2.0, 2.0))
        assert vg.has_isotropic_voxels() is expected
