"""The forward projector's line kernel (column-coherent geometries, planes)
against the FP64 oracle at the edges of its tiles and windows: relative L2
<= 1e-5, pointwise <= 1e-4 * max|ref| (the parity bar)."""
import numpy as np
import pytest

import oracle
from conftest import assert_parity

pytestmark = pytest.mark.gpu

kk = pytest.importorskip("kernelkit")
from kernelkit import _native, workloads  # noqa: E402


def _dev(a):
    import torch
    return torch.from_numpy(np.ascontiguousarray(a, dtype=np.float32)).cuda()


def _case(shape, angles, rows, cols, spacing, sod=None):
    """Rows about ``spacing`` voxels apart at the volume's centre."""
    sod = sod or 4.0 * max(shape)
    pgs = workloads.circular_geometry(angles, sod, 0.5 * sod, rows, cols,
                                      1.5 * spacing)
    vg = kk.resolve_volume_geometry(shape=shape, voxel_size=1.0)
    rng = np.random.default_rng(rows)
    vol = rng.standard_normal(shape).astype(np.float32)
    return pgs, vg, vol


# (volume, angles, rows, columns, spacing): rows per thread 1 to 4, windows of
# 1 to 4 chunks, detectors beyond and inside the volume, columns that do not
# fill a workgroup, one-voxel volumes, rows at the edges of the groups of 64
SIZES = [
    ((20, 24, 33), 8, 129, 9, 0.3),
    ((20, 24, 90), 8, 128, 6, 0.7),
    ((16, 20, 130), 8, 192, 5, 0.7),
    ((16, 20, 150), 8, 193, 4, 0.75),
    ((16, 12, 200), 8, 256, 3, 0.8),
    ((16, 12, 100), 8, 257, 1, 0.8),
    ((12, 16, 300), 8, 320, 2, 1.0),
    ((12, 16, 340), 6, 200, 2, 1.7),
    ((24, 20, 1), 8, 150, 7, 0.6),
    ((1, 24, 40), 8, 150, 7, 0.6),
    ((24, 1, 40), 8, 150, 7, 0.6),
]


@pytest.mark.parametrize("size", SIZES, ids=lambda s: "x".join(map(str, s[0]))
                         + f"-{s[2]}x{s[3]}@{s[4]}")
def test_line_kernel_matches_oracle(size, device):
    pgs, vg, vol = _case(*size)
    A = kk.XrayTransform(pgs, vg)
    assert A.projector.kernel.reads_planes
    y = A(_dev(vol))
    ref = oracle.cone_fp(vol, pgs, vg)
    assert_parity(y.cpu().numpy(), ref)
    # accumulating, and through a table of per-angle outputs
    y2 = A(_dev(vol), out=y.clone(), additive=True)
    assert_parity(y2.cpu().numpy(), 2 * ref)
    parts = [y.new_empty(y.shape[1:]) for _ in pgs]
    A.projector.projections = parts
    A.projector()
    for p, q in zip(parts, y):
        assert bool((p == q).all())


def test_volume_axis_orders_and_detector_off_the_volume(device):
    pgs, vg, vol = _case((20, 28, 60), 12, 200, 20, 0.8)
    ref = oracle.cone_fp(vol, pgs, vg)
    A = kk.XrayTransform(pgs, vg, volume_axes=(2, 1, 0),
                         projection_axes=(1, 0, 2))
    y = A(_dev(vol.transpose(2, 1, 0)))
    assert_parity(y.cpu().numpy(), ref.transpose(1, 0, 2))


def test_texture_keeps_the_set_volume_across_geometries(device):
    """The volume as set is what a geometry set later projects, also where
    that one reads pairs; in-place changes of the source do not show."""
    import torch
    pgs, vg, vol = _case((24, 24, 60), 12, 150, 20, 0.8)
    tilted = workloads.circular_geometry(12, 96.0, 48.0, 150, 20, 1.2,
                                         tilt_deg=2.0)
    A = kk.XrayTransform(pgs, vg)
    x = _dev(vol)
    p = A.projector
    p.volume = x
    assert p._texture.planes is not None
    x.zero_()
    p.projection_geometry = tilted
    assert p._texture.planes is None
    p.projections = torch.empty((12, 150, 20), device="cuda")
    p()
    assert_parity(p.projections.cpu().numpy(),
                  oracle.cone_fp(vol, tilted, vg))
    p.projection_geometry = pgs      # pairs again hold the volume
    p()
    assert_parity(p.projections.cpu().numpy(), oracle.cone_fp(vol, pgs, vg))


def test_extreme_values_follow_the_gather_kernel(device):
    """Largest finite, infinite and NaN voxels reach the same pixels as in
    the gather kernel (pairs)."""
    pgs, vg, vol = _case((16, 16, 70), 8, 150, 12, 0.8)
    vol[3, 4, 10] = np.finfo(np.float32).max / 64
    vol[8, 8, 30] = np.inf
    vol[12, 5, 50] = np.nan
    A = kk.XrayTransform(pgs, vg)
    K = A.projector.kernel
    y = A(_dev(vol)).cpu().numpy()
    tex = A.projector._texture
    lib = _native.lib()
    import torch
    out = torch.empty(y.shape, device="cuda")
    _native.check(lib.kk_cone_fp(
        K._plan.ptr, _native._vp(tex.ptr), _native._vp(out.data_ptr()),
        _native.i64(out.stride()), y.shape[1], y.shape[2], 0,
        _native.stream_ptr()))
    ref = out.cpu().numpy()
    assert np.array_equal(np.isnan(y), np.isnan(ref))
    fin = np.isfinite(ref)
    assert np.array_equal(fin, np.isfinite(y))
    np.testing.assert_allclose(y[fin], ref[fin], rtol=1e-5,
                               atol=1e-5 * np.abs(ref[fin]).max())
