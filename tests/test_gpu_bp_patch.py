"""The backprojector's patch kernel (circular orbits, planes) against the FP64
oracle at the edges of its tiles and patches: relative L2 <= 1e-5, pointwise
<= 1e-4 * max|ref| (the parity bar)."""
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


def _case(shape, angles, rows, cols, pixel, sod=None, **pert):
    sod = sod or 4.0 * max(shape)
    pgs = workloads.circular_geometry(angles, sod, 0.5 * sod, rows, cols,
                                      pixel, **pert)
    vg = kk.resolve_volume_geometry(shape=shape, voxel_size=1.0)
    y = np.random.default_rng(rows + cols).standard_normal(
        (angles, rows, cols)).astype(np.float32)
    return pgs, vg, y


# (volume, angles, rows, columns, pixel): tiles that do not divide, one voxel,
# detectors smaller than the volume's projection and of one pixel, fewer
# angles than parts, more than one batch of 64 patches, patches of up to 64
# columns, and tile counts on either side of the parts' rule
SIZES = [
    ((16, 16, 16), 5, 40, 40, 1.0),
    ((17, 33, 15), 3, 30, 50, 1.2),
    ((1, 1, 1), 4, 9, 9, 1.0),          # (the run reaches far past: pairs)
    ((1, 1, 1), 4, 9, 9, 1.0, 64.0),
    ((40, 24, 70), 66, 33, 21, 1.5),
    ((40, 24, 70), 6, 1, 1, 1.5),
    ((48, 48, 48), 260, 20, 90, 1.1),
    ((64, 40, 30), 2, 150, 150, 0.6),
    ((128, 128, 72), 7, 90, 170, 1.3),
    ((144, 130, 200), 5, 180, 190, 1.4),
]


@pytest.mark.parametrize("size", SIZES, ids=lambda s: "x".join(map(str, s[0]))
                         + f"-{s[1]}-{s[2]}x{s[3]}@{s[4]}")
def test_patch_kernel_matches_oracle(size, device):
    pgs, vg, y = _case(*size)
    A = kk.XrayTransform(pgs, vg)
    assert A.backprojector.kernel.reads_planes == (size[0] != (1, 1, 1)
                                                   or len(size) > 5)
    x = A.T(_dev(y))
    ref = oracle.cone_bp(y, pgs, vg)
    assert_parity(x.cpu().numpy(), ref)
    np.testing.assert_array_equal(A.backprojector.projections.cpu().numpy(), y)
    x2 = A.T(_dev(y), out=x.clone(), additive=True)
    assert_parity(x2.cpu().numpy(), 2 * ref)


@pytest.mark.parametrize("pert", [
    dict(wobble_deg=1.0, drift_px=3.0),
    dict(wobble_deg=12.0, tilt_deg=30.0, drift_px=2.0)],
    ids=["wobble", "strong"])
@pytest.mark.parametrize("size", SIZES, ids=lambda s: "x".join(map(str, s[0]))
                         + f"-{s[1]}-{s[2]}x{s[3]}@{s[4]}")
def test_general_geometries_match_oracle(size, pert, device):
    """The same sizes on wobbling orbits (with the kernel that the plan
    picks; all but the largest patches of the strong ones fit)."""
    size = (*size[:5], size[5] if len(size) > 5 else 5.0 * max(size[0]))
    pgs, vg, y = _case(*size, **pert)
    A = kk.XrayTransform(pgs, vg)
    assert A.backprojector.kernel.reads_planes or size[0] == (1, 1, 1) or \
        pert["wobble_deg"] > 1
    x = A.T(_dev(y))
    ref = oracle.cone_bp(y, pgs, vg)
    assert_parity(x.cpu().numpy(), ref)
    x2 = A.T(_dev(y), out=x.clone(), additive=True)
    assert_parity(x2.cpu().numpy(), 2 * ref)


def test_mixed_angles_match_oracle(device):
    """Circular, tilted and wobbling angles in one plan."""
    pgs, vg, y = _case((40, 36, 33), 12, 50, 60, 1.1)
    pgs = pgs[:4] + _case((40, 36, 33), 12, 50, 60, 1.1, tilt_deg=3.0)[0][
        4:8] + _case((40, 36, 33), 12, 50, 60, 1.1, wobble_deg=2.0)[0][8:]
    A = kk.XrayTransform(pgs, vg)
    assert A.backprojector.kernel.reads_planes
    assert_parity(A.T(_dev(y)).cpu().numpy(), oracle.cone_bp(y, pgs, vg))


def test_axis_orders_and_texture_across_geometries(device):
    """Arrays in other axis orders; projections as set are what a geometry
    set later backprojects, also where that one reads pairs."""
    import torch
    pgs, vg, y = _case((40, 28, 36), 12, 50, 60, 1.1)
    ref = oracle.cone_bp(y, pgs, vg)
    A = kk.XrayTransform(pgs, vg, volume_axes=(2, 1, 0),
                         projection_axes=(1, 0, 2))
    x = A.T(_dev(y.transpose(1, 0, 2)))
    assert_parity(x.cpu().numpy(), ref.transpose(2, 1, 0))
    A = kk.XrayTransform(pgs, vg)
    p, src = A.backprojector, _dev(y)
    p.projections = src
    assert p._textures.planes is not None
    src.zero_()
    tilted = workloads.circular_geometry(12, 160.0, 80.0, 50, 60, 1.1,
                                         tilt_deg=2.0)
    p.projection_geometry = tilted
    assert p._textures.planes is None
    p.volume = torch.empty((40, 28, 36), device="cuda")
    p()
    assert_parity(p.volume.cpu().numpy(), oracle.cone_bp(y, tilted, vg))


def test_sirt_update_and_residual_match_the_pair_kernels(device):
    """The update epilogue and the residual planes, against the pair kernels'
    forms of both (same operations up to the row's rounding)."""
    import torch
    pgs, vg, y = _case((40, 28, 36), 12, 50, 60, 1.1)
    A = kk.XrayTransform(pgs, vg)
    K, lib, vp = A.backprojector.kernel, _native.lib(), _native._vp
    n, rows, cols = y.shape
    rng = np.random.default_rng(1)
    p, R = _dev(rng.standard_normal(y.shape)), _dev(rng.uniform(0, 1, y.shape))
    yd, C = _dev(y), _dev(rng.uniform(0, 1e-3, vg.shape))
    mask = _dev(rng.uniform(0, 1, vg.shape) > 0.3)
    x = [_dev(np.ones(vg.shape)) for _ in range(2)]
    from kernelkit.kernel import ProjectionTexture
    tex = [ProjectionTexture(n, rows, cols, like=yd) for _ in range(2)]
    st = _native.stream_ptr()
    src = (vp(p.data_ptr()), _native.i64(p.stride()), vp(yd.data_ptr()),
           _native.i64(yd.stride()), vp(R.data_ptr()),
           _native.i64(R.stride()), n, rows, cols)
    _native.check(lib.kk_residual_to_bp_planes(
        *src, vp(tex[0].hold_planes()), st))
    _native.check(lib.kk_residual_to_bp_texture(*src, vp(tex[1].ptr), st))
    assert torch.equal(tex[0].values(), tex[1].values())

    def args(t, v):
        return (K._plan.ptr, vp(t), n, rows, cols, vp(v.data_ptr()),
                _native.i32(vg.shape), _native.i64(v.stride()),
                vp(C.data_ptr()), _native.i64(C.stride()),
                vp(mask.data_ptr()), _native.i64(mask.stride()), 0.2, 1.5, 1,
                1)
    _native.check(lib.kk_sirt_bp_update_planes(
        *args(tex[0].planes, x[0]), 1.0, st))
    _native.check(lib.kk_sirt_bp_update(
        *args(tex[1].ptr, x[1]), None, 0, 1.0, st))
    a, b = x[0].cpu().numpy(), x[1].cpu().numpy()
    assert a.min() >= np.float32(0.2) and a.max() <= np.float32(1.5)
    np.testing.assert_allclose(a, b, rtol=2e-6, atol=2e-6)
    assert torch.equal(tex[0].data, tex[1].data)   # planes made pairs


def test_extreme_values_follow_the_pair_kernel(device):
    pgs, vg, y = _case((20, 20, 20), 6, 40, 40, 1.0)
    y[1, 7, 9] = np.finfo(np.float32).max / 64
    y[2, 20, 20] = np.inf
    y[3, 30, 11] = np.nan
    A = kk.XrayTransform(pgs, vg)
    x = A.T(_dev(y)).cpu().numpy()
    p = A.backprojector
    p._textures.data           # pairs now
    p()
    ref = p.volume.cpu().numpy()
    assert np.array_equal(np.isnan(x), np.isnan(ref))
    fin = np.isfinite(ref)
    assert np.array_equal(fin, np.isfinite(x))
    np.testing.assert_allclose(x[fin], ref[fin], rtol=1e-5,
                               atol=1e-5 * np.abs(ref[fin]).max())
