"""Threaded copies of device results into host memory (kk_copy_to_host):
bytes equal around the sizes where pieces and workers begin."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

kk = pytest.importorskip("kernelkit")
from kernelkit import _native, device as dev  # noqa: E402

PIECE = 2 << 20


@pytest.mark.parametrize("n", [1, PIECE // 4 - 1, PIECE // 4, PIECE // 4 + 1,
                               3 * PIECE // 4 + 7, 6 * PIECE // 4,
                               13 * PIECE // 4 + 5])
def test_bytes_equal(n, device):
    import torch
    x = torch.randn(n, device="cuda")
    out = np.full(n + 2, np.float32(7))
    _native.check(_native.lib().kk_copy_to_host(
        out[1:].ctypes.data, x.data_ptr(), 4 * n, _native.stream_ptr()))
    np.testing.assert_array_equal(out[1:-1], x.cpu().numpy())
    assert out[0] == 7 and out[-1] == 7


def test_to_host_orders_after_the_stream_and_fills_out(device):
    import torch
    s = torch.cuda.Stream()
    with torch.cuda.stream(s):
        x = torch.zeros((128, 128, 160), device="cuda")
        for _ in range(50):
            x += 1
        a = dev.to_host(x)
        out = np.zeros(x.shape, np.float32)
        assert dev.to_host(x, out) is out
        wide = np.zeros((2,) + tuple(x.shape))
        dev.to_host(x, wide)
    assert (a == 50).all() and (out == 50).all() and (wide == 50).all()
    v = dev.to_host(x.transpose(0, 2)[::2])
    assert v.shape == (80, 128, 128) and (v == 50).all()
    d = dev.from_host(np.arange(3 << 20, dtype=np.float32))
    np.testing.assert_array_equal(d.get(), np.arange(3 << 20))


def test_bad_arguments():
    lib = _native.lib()
    assert lib.kk_copy_to_host(None, None, 0, None) == _native.KK_OK
    assert lib.kk_copy_to_host(None, None, 4, None) == _native.KK_ERR_INVALID
    assert lib.kk_copy_to_host(None, None, -1, None) == _native.KK_ERR_INVALID
