"""Forward projection along an axis of 16384 slices: sample coordinates at its
far end are as good as anywhere (rays just inside the low face, whose weights
are the coordinates' own distance from it)."""
import numpy as np
import pytest

import oracle

pytestmark = pytest.mark.gpu

kk = pytest.importorskip("kernelkit")
from kernelkit.batch import ConeBatch  # noqa: E402
from kernelkit.geom.proj import Detector, ProjectionGeometry  # noqa: E402

LONG, END = 16384, 64        # slices, and those with values: one end's
NB, NC = 8, 40


def _geometry(end, tilt=0.0):
    """Rays 0.008 to 0.05 voxel inside the volume's low z face at one end of the
    x axis; ``tilt`` (degrees, in the detector's plane) makes the b coordinate
    depend on the row."""
    det = Detector(rows=128, cols=9, pixel_height=0.0004, pixel_width=0.3)
    x_end = (0.5 * LONG - 0.5 * END) * (1 if end else -1)
    sod, odd = 40000.0, 20000.0
    f = (x_end + sod) / (sod + odd)
    zs = -0.5 * NC - 0.5 + 0.03
    zd = zs + (0.0285 - 0.03) / f
    c, s = np.cos(np.deg2rad(tilt)), np.sin(np.deg2rad(tilt))
    return [ProjectionGeometry([-sod, 0.01 * k, zs], [odd, 0.013 * k, zd], det,
                               u=[0.0, c, s], v=[0.0, -s, c])
            for k in range(-6, 7)]


@pytest.mark.parametrize("batched", [False, True])
@pytest.mark.parametrize("tilt", [0.0, 1e-5])
@pytest.mark.parametrize("end", [0, 1])
def test_both_ends(end, tilt, batched, device):
    import torch
    pgs = _geometry(end, tilt)
    rng = np.random.default_rng(end)
    v = rng.uniform(0.5, 1.5, (END, 1, 1)).astype(np.float32)
    part = np.broadcast_to(v, (END, NB, NC))
    first = (LONG - END) * end
    x = torch.zeros((LONG, NB, NC), device="cuda")
    x[first:first + END] = torch.from_numpy(part.copy())
    vg = kk.resolve_volume_geometry(shape=(LONG, NB, NC), voxel_size=1.0)
    if batched:
        B = ConeBatch([(pgs, vg)] * 2)
        got = B.fp([x, 2.0 * x], tune=False)[0]
    else:
        got = kk.XrayTransform(pgs, vg)(x)
    got = got.cpu().numpy().astype(np.float64)
    lo = first - 0.5 * LONG
    ref = oracle.cone_fp(part, pgs, kk.resolve_volume_geometry(
        shape=(END, NB, NC), extent_min=(lo, -0.5 * NB, -0.5 * NC),
        extent_max=(lo + END, 0.5 * NB, 0.5 * NC)))
    assert (ref > 0).mean() > 0.8
    # a coordinate 2^-23 voxel off, over the least depth; 64 float32 additions;
    # a few roundings each
    bound = 2.0 ** -23 / 0.008 + (END + 10) * 2.0 ** -24
    worst = float((np.abs(got - ref)[ref > 0] / ref[ref > 0]).max())
    assert worst <= bound, (worst, bound)
