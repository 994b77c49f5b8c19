"""Host side of the forward projector's line kernel: the bound on the rows'
c spacing that sizes its windows, and its fixed-point coordinates."""
import numpy as np
import pytest

kk = pytest.importorskip("kernelkit")
from kernelkit import _native, workloads  # noqa: E402
from kernelkit.kernels.cone_fp import RayDrivenConeFP  # noqa: E402

FRAME = {0: (0, 1, 2), 1: (1, 0, 2), 2: (2, 1, 0)}


def _spacing(pgs, vg, rows, cols):
    p = RayDrivenConeFP.geoms2params(pgs, vg)
    a = np.ascontiguousarray(np.stack([np.asarray(v) for v in p]))
    axes = np.ascontiguousarray(p.ray_axes, dtype=np.int32)
    out = np.zeros(2)
    _native.check(_native.lib().kk_fp_line_spacing(
        _native.f64_ptr(a), a.shape[1], _native.i32_ptr(axes), rows, cols,
        _native.i32(vg.shape), _native.f64(vg.voxel_size),
        _native.f64_ptr(out)))
    return a, axes, out


@pytest.mark.parametrize("shape,rows,cols,sod,odd,pixel", [
    ((64, 64, 64), 80, 96, 150.0, 75.0, 1.0),
    ((33, 71, 20), 64, 200, 90.0, 200.0, 2.5),
    ((48, 16, 40), 129, 31, 60.0, 30.0, 3.0),
])
def test_spacing_bound_covers_every_workgroup_slice(shape, rows, cols, sod,
                                                    odd, pixel):
    """No sample of a column at a slice that any of the workgroup's four
    columns needs (two slices of slack) is further from the next row's than
    the bound."""
    pgs = workloads.circular_geometry(24, sod, odd, rows, cols, pixel)
    vg = kk.resolve_volume_geometry(shape=shape, voxel_size=1.0)
    a, axes, out = _spacing(pgs, vg, rows, cols)
    assert out[0] >= out[1] > 0
    worst = 0.0
    for k in range(a.shape[1]):
        A, B, C = FRAME[int(axes[k])]
        s, d0, U, V = (a[3 * i:3 * i + 3, k] for i in range(4))
        col = np.arange(cols) + 0.5
        D = [d0[t] + col * U[t] + 0.5 * V[t] - s[t] for t in range(3)]
        i = np.arange(shape[A])[:, None] + 0.5 - 0.5 * shape[A] - s[A]
        t = i / D[A]
        xb = s[B] + t * D[B] + 0.5 * shape[B] - 0.5
        inside = (xb > -1) & (xb < shape[B])
        for c0 in range(0, cols, 4):
            need = np.flatnonzero(inside[:, c0:c0 + 4].any(1))
            if need.size == 0:
                continue
            lo, hi = max(0, need[0] - 2), min(shape[A], need[-1] + 3)
            worst = max(worst, float(np.abs(
                V[C] * t[lo:hi, c0:c0 + 4]).max()))
    assert worst <= out[0]


def test_spacing_refuses_other_geometries():
    vg = kk.resolve_volume_geometry(shape=(32, 32, 32), voxel_size=1.0)
    for kw in (dict(tilt_deg=1.0), dict(wobble_deg=1.0)):
        pgs = workloads.circular_geometry(8, 100.0, 50.0, 40, 40, 1.0, **kw)
        assert _spacing(pgs, vg, 40, 40)[2][0] < 0
    # the source among the slices
    pgs = workloads.circular_geometry(8, 10.0, 50.0, 40, 40, 1.0)
    assert _spacing(pgs, vg, 40, 40)[2][0] < 0


def test_fixed_point_steps_stay_below_float32_weights():
    """x(i) = a i + b stepped in 32.32 fixed point: element and weight are
    those of the float64 coordinate within 2^-33 per slice, below half a
    float32 ulp of a weight in [1/2, 1) for 256 slices and below 2^-23 at
    1024."""
    rng = np.random.default_rng(0)
    a = rng.uniform(-0.6, 0.6, 200)
    b = rng.uniform(-50.0, 1100.0, 200)
    X = np.floor(b * 2.0 ** 32).astype(np.int64)
    S = np.floor(a * 2.0 ** 32).astype(np.int64)
    for n in (256, 1024):
        err = np.abs((X + S * n) / 2.0 ** 32 - (a * n + b))
        assert err.max() <= (n + 2) * 2.0 ** -32


def test_spacing_refuses_axes_longer_than_its_steps_are_good_for():
    """Steps of 2^-32 voxel, rounded, from the middle slice: 2^-23 voxel off at
    the ends of 2048 slices."""
    for n, fine in ((2048, True), (2049, False)):
        pgs = workloads.circular_geometry(1, 3.0 * n, 1.5 * n, 70, 20, 1.0)
        vg = kk.resolve_volume_geometry(shape=(n, 8, 40), voxel_size=1.0)
        assert bool(_spacing(pgs, vg, 70, 20)[2][0] > 0) is fine
