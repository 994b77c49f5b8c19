"""The forward projector's gather kernel (tilted and wobbling geometries, and
batches) against the FP64 oracle at the edges of its wavefronts and of its
fixed-point coordinates: relative L2 <= 1e-5, pointwise <= 1e-4 * max|ref| (the
parity bar)."""
import numpy as np
import pytest

import oracle
from conftest import assert_parity

pytestmark = pytest.mark.gpu

kk = pytest.importorskip("kernelkit")
from kernelkit import workloads  # noqa: E402
from kernelkit.batch import ConeBatch  # noqa: E402
from kernelkit.geom.proj import Detector, ProjectionGeometry  # noqa: E402

PERT = dict(tilt_deg=3.0, wobble_deg=2.0, drift_px=2.0)


def _dev(a):
    import torch
    return torch.from_numpy(np.ascontiguousarray(a, dtype=np.float32)).cuda()


def _problem(shape, angles, rows, cols, pixel, seed=0):
    pgs = workloads.circular_geometry(angles, 150.0, 75.0, rows, cols, pixel,
                                      seed=seed, **PERT)
    vg = kk.resolve_volume_geometry(shape=shape, voxel_size=1.0)
    x = np.random.default_rng(rows * cols).uniform(size=shape)
    return pgs, vg, x.astype(np.float32)


# rows around the wavefronts' 1, 2, 4, 8, 16 and 32 rows and bands of them,
# columns around the workgroups', volumes of one slice or voxel
SIZES = [((20, 22, 18), 5, r, c, 1.5) for r, c in
         [(1, 1), (1, 300), (2, 33), (3, 8), (5, 9), (15, 17), (16, 7),
          (17, 31), (31, 40), (32, 8), (33, 9), (64, 20), (139, 5)]] + \
    [((1, 1, 1), 3, 9, 9, 0.5), ((1, 30, 30), 4, 20, 20, 1.5),
     ((40, 1, 9), 4, 20, 20, 1.5), ((90, 80, 70), 9, 65, 70, 2.0)]


@pytest.mark.parametrize("size", SIZES, ids=str)
def test_gather_kernel_matches_oracle(size, device):
    pgs, vg, x = _problem(*size)
    A = kk.XrayTransform(pgs, vg)
    assert not A.projector.kernel.reads_planes
    y = A(_dev(x))
    ref = oracle.cone_fp(x.astype(np.float64), pgs, vg)
    assert_parity(y.cpu().numpy(), ref)
    y2 = A(_dev(x), out=y.clone(), additive=True)
    assert_parity(y2.cpu().numpy(), 2 * ref)


def test_batches_give_the_single_launches_bits(device):
    import torch
    probs = [_problem(*s, seed=k) for k, s in enumerate(SIZES)]
    B = ConeBatch([(pgs, vg) for pgs, vg, _ in probs])
    vols = [_dev(x) for _, _, x in probs]
    for y, (pgs, vg, _), v in zip(B.fp(vols, tune=False), probs, vols):
        assert torch.equal(y, kk.XrayTransform(pgs, vg)(v)), vg.shape


@pytest.mark.parametrize("off", [0.0, 1e-12, -1e-9, 1e-7, -3e-5])
@pytest.mark.parametrize("x0", [-40.0, 0.0, 0.5])
def test_rays_parallel_to_the_slices(off, x0, device):
    """Rays whose slope is too large for the fixed-point coordinates, from a
    source outside the volume, in a slice and between two."""
    det = Detector(rows=5, cols=41, pixel_height=0.7, pixel_width=1.0)
    s = np.array([x0, 0.25, -0.5])
    u = np.array([-1.0, 0.0, 0.0])
    v = np.array([0.0, 0.6, 0.8])
    # the rays of column 34 run along the slices, but for `off`
    pgs = [ProjectionGeometry(s, s + [14.0 + off, 12.0, 0.0], det, u=u, v=v)]
    vg = kk.resolve_volume_geometry(shape=(31, 27, 20), voxel_size=1.0)
    x = np.random.default_rng(3).uniform(size=(31, 27, 20))
    x = x.astype(np.float32)
    A = kk.XrayTransform(pgs, vg)
    with np.errstate(all="ignore"):   # exactly parallel: skipped, 0
        ref = np.nan_to_num(oracle.cone_fp(x.astype(np.float64), pgs, vg,
                                           axes=[0]))
    got = A(_dev(x)).cpu().numpy()
    assert A.projector.kernel.frame_mask == 1
    assert not A.projector.kernel.reads_planes
    steep = np.zeros(ref.shape, dtype=bool)
    steep[:, :, 34] = True
    assert_parity(np.where(steep, 0, got), np.where(steep, 0, ref))
    # a slope a puts the sample within a * 2^-52 * 31 slices of its place
    if off == 0.0 or abs(off) >= 1e-9:
        np.testing.assert_allclose(got[steep], ref[steep], rtol=1e-3)
