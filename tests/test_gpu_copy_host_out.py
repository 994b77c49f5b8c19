"""Device results of several megabytes into host arrays that are more than
their bytes: what an assignment means to them holds."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

kk = pytest.importorskip("kernelkit")
from kernelkit import device as dev  # noqa: E402

SHAPE = (5, 512, 513)    # above the threaded copy's threshold


def test_masked_arrays_keep_their_masks(device):
    import torch
    x = torch.rand(SHAPE, device="cuda")
    host = x.cpu().numpy()
    for hard in (False, True):
        def made():
            m = np.zeros(SHAPE, bool)
            m[:, ::2] = True
            return np.ma.masked_array(np.full(SHAPE, 7, np.float32), mask=m,
                                      hard_mask=hard)
        want, got = made(), made()
        want[...] = host
        assert dev.to_host(x, got) is got
        np.testing.assert_array_equal(np.ma.getmaskarray(got),
                                      np.ma.getmaskarray(want))
        np.testing.assert_array_equal(got.data, want.data)


def test_plain_and_mapped_arrays(device, tmp_path):
    import torch
    x = torch.rand(SHAPE, device="cuda")
    plain = np.zeros(SHAPE, np.float32)
    mapped = np.memmap(tmp_path / "out", np.float32, "w+", shape=SHAPE)
    for out in (plain, mapped):
        assert dev.to_host(x, out) is out
        np.testing.assert_array_equal(out, x.cpu().numpy())


def test_negative_views(device):
    """A view whose bytes are the values' negatives."""
    import torch
    x = torch._neg_view(torch.rand(SHAPE, device="cuda"))
    out = np.zeros(SHAPE, np.float32)
    assert dev.to_host(x, out) is out
    np.testing.assert_array_equal(out, x.cpu().numpy())
    np.testing.assert_array_equal(dev.to_host(x), out)
    assert (out <= 0).all() and (out < 0).any()
