"""Which layout circular orbits read (planes for the line and patch kernels,
pairs for the general ones) on either side of the rules' lines, each against
the FP64 oracle: relative L2 <= 1e-5, pointwise <= 1e-4 * max|ref| (the parity
bar)."""
import numpy as np
import pytest

import oracle
from conftest import assert_parity

pytestmark = pytest.mark.gpu

kk = pytest.importorskip("kernelkit")
from kernelkit import workloads  # noqa: E402


def _dev(a):
    import torch
    return torch.from_numpy(np.ascontiguousarray(a, dtype=np.float32)).cuda()


def _operator(shape, angles, rows, cols, pixel, **kw):
    sod = 3.0 * max(shape)
    pgs = workloads.circular_geometry(angles, sod, 0.5 * sod, rows, cols,
                                      pixel, **kw)
    vg = kk.resolve_volume_geometry(shape=shape, voxel_size=1.0)
    return kk.XrayTransform(pgs, vg), pgs, vg


# (volume, angles, rows, columns, pixel, planes): few rows far apart, up to 32
# and more of them; few and many workgroups of a volume that the caches hold
# and of one that they do not
@pytest.mark.parametrize("case", [
    ((66, 60, 9), 6, 3, 30, 3.0, False),
    ((40, 36, 40), 6, 32, 25, 2.4, False),
    ((40, 36, 90), 5, 65, 20, 3.0, True),
    ((80, 70, 100), 3, 160, 30, 1.0, False),
    ((80, 70, 100), 70, 150, 64, 1.1, True),
    ((250, 240, 200), 2, 300, 90, 1.0, False),
    ((250, 240, 200), 3, 300, 200, 1.0, True),
], ids=str)
def test_forward(case, device):
    *args, planes = case
    A, pgs, vg = _operator(*args)
    assert A.projector.kernel.reads_planes is planes
    vol = np.random.default_rng(3).standard_normal(args[0]).astype(np.float32)
    y = A(_dev(vol))
    k = [0, len(pgs) // 2, len(pgs) - 1]
    assert_parity(y.cpu().numpy()[k],
                  oracle.cone_fp(vol, [pgs[i] for i in k], vg))


# volumes of one layer of tiles, half of it empty or not, of fewer tiles than
# CUs and of more
@pytest.mark.parametrize("kw", [{}, dict(wobble_deg=0.5)],
                         ids=["circular", "wobble"])
@pytest.mark.parametrize("shape,planes", [
    ((256, 250, 8), True), ((272, 250, 8), False), ((272, 250, 9), True),
    ((272, 258, 1), False)], ids=str)
def test_backprojection(shape, planes, kw, device):
    A, pgs, vg = _operator(shape, 4, 14, 300, 1.2, **kw)
    assert A.backprojector.kernel.reads_planes is planes
    y = np.random.default_rng(4).uniform(size=(4, 14, 300)).astype(np.float32)
    x = A.T(_dev(y))
    assert_parity(x.cpu().numpy(), oracle.cone_bp(y, pgs, vg))
