"""Kernel classes of a program's own, written to the interface that projectors
and ``algo.bp`` ask for: parameters, textures and calls, nothing about
planes."""
import numpy as np
import pytest

kk = pytest.importorskip("kernelkit")
from kernelkit import _native, algo, device as dev, workloads  # noqa: E402
from kernelkit.projector import BackProjector, ForwardProjector  # noqa: E402


class _StubLibrary:
    def __getattr__(self, name):
        if not name.startswith("kk_"):
            raise AttributeError(name)

        def call(*args):
            if name.endswith("_elems"):
                return 64
            if name in ("kk_malloc", "kk_filter_create"):
                args[0]._obj.value = 0   # nothing to free
            return _native.KK_OK
        return call


class _Kernel:
    """Neither ``reads_planes`` nor a ``pairs`` argument."""

    volume_axes = (0, 1, 2)
    projection_axes = (0, 1, 2)
    is_compiled = True
    frame_mask = 0b011

    def __init__(self):
        self.log = []

    def compile(self, **kw):
        pass

    def geoms2params(self, pgs, vg):
        return np.zeros(12 * len(pgs))

    def set_params(self, params, pgs=None, vg=None):
        self.log.append("params")

    def projection_texture(self, projections, texture=None):
        self.log.append("texture")
        return ("texture of", projections)

    def __call__(self, *args, **kw):
        self.log.append("call")


@pytest.fixture
def stub(monkeypatch):
    s = _StubLibrary()
    monkeypatch.setattr(_native, "lib", lambda: s)
    monkeypatch.setattr(_native, "_lib", s)


def _array(shape):
    return dev.DeviceArray(shape, np.float32, ptr=0x900000, device=0)


def _geometry():
    return (workloads.circular_geometry(3, 40.0, 20.0, 5, 6, 1.0),
            kk.resolve_volume_geometry(shape=(4, 4, 4), voxel_size=1.0))


def test_backprojector(stub):
    pgs, vg = _geometry()
    K = _Kernel()
    P = BackProjector(kernel=K)
    P.volume_geometry = vg
    P.projection_geometry = pgs
    P.projections = _array((3, 5, 6))
    P.projection_geometry = pgs[::-1]
    P.volume = _array((4, 4, 4))
    P()
    assert K.log == ["params", "texture", "params", "call"]


def test_forward_projector(stub):
    pgs, vg = _geometry()
    K = _Kernel()
    P = ForwardProjector(kernel=K)
    P.volume_geometry = vg
    P.projection_geometry = pgs
    P.volume = _array((4, 4, 4))
    P.projection_geometry = pgs[::-1]
    P.projections = _array((3, 5, 6))
    P()
    assert K.log == ["params", "params", "call"]


def test_bp_with_a_filter(stub, monkeypatch):
    pgs, vg = _geometry()
    K = _Kernel()
    monkeypatch.setattr(algo, "_to_host", lambda t, out=None: t)
    monkeypatch.setattr(algo, "default_device", lambda: None)
    algo.bp(_array((3, 5, 6)), pgs, vg, filter="ramlak", kernel=K)
    assert K.log[-1] == "call"
