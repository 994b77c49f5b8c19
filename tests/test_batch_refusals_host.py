"""What a batch refuses before it launches anything, shown with a stub in the
library's place."""
import numpy as np
import pytest

kk = pytest.importorskip("kernelkit")
from kernelkit import _native, device as dev, workloads  # noqa: E402
from kernelkit.batch import ConeBatch  # noqa: E402


class _StubLibrary:
    def __init__(self):
        self.calls = []

    def __getattr__(self, name):
        if not name.startswith("kk_"):
            raise AttributeError(name)

        def call(*args):
            self.calls.append(name)
            if name.endswith("_elems"):
                return 64
            if name.endswith("_create") or name == "kk_malloc":
                args[0]._obj.value = 0   # nothing to free
            return _native.KK_OK
        return call


@pytest.fixture
def stub(monkeypatch):
    s = _StubLibrary()
    monkeypatch.setattr(_native, "lib", lambda: s)
    monkeypatch.setattr(_native, "_lib", s)
    return s


@pytest.mark.parametrize("odd_one", [0, 1])
def test_sirt_of_anisotropic_voxels(stub, odd_one):
    """The backprojector does not take them, whichever way it is reached."""
    pgs = workloads.circular_geometry(3, 40.0, 20.0, 5, 6, 1.0)
    sizes = [(1.0, 1.0, 1.0)] * 2
    sizes[odd_one] = (1.0, 1.0, 2.0)
    B = ConeBatch([(pgs, kk.resolve_volume_geometry(shape=(4, 4, 4),
                                                    voxel_size=v))
                   for v in sizes])
    ys = [dev.DeviceArray((3, 5, 6), np.float32, ptr=0x900000, device=0)] * 2
    with pytest.raises(NotImplementedError, match="anisotropic"):
        B.sirt_state(ys)
    assert not [c for c in stub.calls if c.startswith("kk_batch_bp")]
