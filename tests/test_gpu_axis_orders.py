"""Every pair of axis orders through the kernels that read planes (lines of
circular forward projections, patches of circular and wobbling
backprojections) and the transposes' kernels, against the FP64 oracle: relative
L2 <= 1e-5, pointwise <= 1e-4 * max|ref| (the parity bar)."""
import itertools

import numpy as np
import pytest

import oracle
from conftest import assert_parity

pytestmark = pytest.mark.gpu

kk = pytest.importorskip("kernelkit")
from kernelkit import workloads  # noqa: E402

ORDERS = list(itertools.permutations((0, 1, 2)))
SHAPE, ANGLES, ROWS, COLS, PIXEL = (40, 36, 90), 5, 65, 20, 3.0


def _dev(a):
    import torch
    return torch.from_numpy(np.ascontiguousarray(a, dtype=np.float32)).cuda()


@pytest.fixture(scope="module", params=[0.0, 0.5], ids=["circular", "wobble"])
def case(request):
    pgs = workloads.circular_geometry(ANGLES, 270.0, 135.0, ROWS, COLS, PIXEL,
                                      wobble_deg=request.param, seed=2)
    vg = kk.resolve_volume_geometry(shape=SHAPE, voxel_size=1.0)
    rng = np.random.default_rng(6)
    vol = rng.standard_normal(SHAPE)
    y = rng.uniform(size=(ANGLES, ROWS, COLS))
    return (pgs, vg, vol, y, oracle.cone_fp(vol, pgs, vg),
            oracle.cone_bp(y, pgs, vg), oracle.cone_fp_transpose(y, pgs, vg),
            request.param == 0.0)


@pytest.mark.parametrize("vaxes", ORDERS, ids=str)
@pytest.mark.parametrize("paxes", ORDERS, ids=str)
def test_axis_orders(case, vaxes, paxes, device):
    pgs, vg, vol, y, fp, bp, fp_t, circular = case
    A = kk.XrayTransform(pgs, vg, volume_axes=vaxes, projection_axes=paxes)
    assert A.projector.kernel.reads_planes is circular
    assert A.backprojector.kernel.reads_planes is True

    got = A(_dev(np.transpose(vol, vaxes))).cpu().numpy()
    assert_parity(np.transpose(got, np.argsort(paxes)), fp)
    yt = _dev(np.transpose(y, paxes))
    got = A.T(yt).cpu().numpy()
    assert_parity(np.transpose(got, np.argsort(vaxes)), bp)
    got = A.matched_T(yt).cpu().numpy()
    assert_parity(np.transpose(got, np.argsort(vaxes)), fp_t)
