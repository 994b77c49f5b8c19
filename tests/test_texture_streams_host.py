"""A texture held as planes, launched by a kernel that reads pairs: the
conversion goes to the launch's stream, shown with a stub in the library's
place (nothing is launched)."""
import numpy as np
import pytest

kk = pytest.importorskip("kernelkit")
from kernelkit import _native, device as dev, kernel, workloads  # noqa: E402
from kernelkit.kernels.cone_bp import VoxelDrivenConeBP  # noqa: E402
from kernelkit.kernels.cone_fp import RayDrivenConeFP  # noqa: E402

STREAM = 0x5000


class _StubLibrary:
    """Records ``(name, stream)`` of the calls that take a stream last."""

    def __init__(self, reads_planes):
        self.reads_planes = reads_planes
        self.calls = []

    def __getattr__(self, name):
        if not name.startswith("kk_"):
            raise AttributeError(name)

        def call(*args):
            if name.endswith("_reads_planes"):
                return self.reads_planes
            if name.endswith("_elems"):
                return 64
            if name == "kk_fp_frame_mask":
                return 0b001
            if name in ("kk_plan_create", "kk_malloc", "kk_event_create"):
                args[0]._obj.value = 0      # nothing to free
            self.calls.append((name, getattr(args[-1], "value", None)
                               if args else None))
            return _native.KK_OK
        return call

    def of(self, *names):
        return [c for c in self.calls if c[0] in names]


@pytest.fixture
def stub(monkeypatch):
    def use(reads_planes):
        s = _StubLibrary(reads_planes)
        monkeypatch.setattr(_native, "lib", lambda: s)
        monkeypatch.setattr(_native, "_lib", s)
        return s
    return use


def _array(shape, ptr=0x900000):
    return dev.DeviceArray(shape, np.float32, ptr=ptr, device=0)


def _geometry(n=3, rows=5, cols=6, shape=(4, 4, 4)):
    pgs = workloads.circular_geometry(n, 40.0, 20.0, rows, cols, 1.0)
    return pgs, kk.resolve_volume_geometry(shape=shape, voxel_size=1.0)


def test_backprojection(stub):
    pgs, vg = _geometry()
    s = stub(1)
    K = VoxelDrivenConeBP()
    K.compile()
    K.set_params(K.geoms2params(pgs, vg), pgs, vg)
    tex = K.projection_texture(_array((3, 5, 6)))
    assert tex.planes is not None
    s.reads_planes = 0          # another volume's patches do not fit
    K.set_params(K.geoms2params(pgs, vg), pgs, vg)
    del s.calls[:]
    for handle in (STREAM, None, STREAM + 1):
        K(tex, _array((4, 4, 4)), vg, stream=handle)
    want = [STREAM, None, STREAM + 1]
    build, launch = "kk_projections_to_bp_texture", "kk_cone_bp"
    assert [h for _, h in s.of(launch)] == want
    # every launch finds its pairs written on its own stream before it
    order = s.of(build, launch)
    for k, (name, handle) in enumerate(order):
        if name == launch:
            assert order[k - 1] == (build, handle)
    assert tex.planes is not None


@pytest.mark.parametrize("as_list", [False, True])
def test_forward_projection(stub, as_list):
    pgs, vg = _geometry()
    s = stub(1)
    K = RayDrivenConeFP()
    K.compile()
    params = K.geoms2params(pgs, vg)
    K.set_params(params, pgs, vg)
    tex = K.volume_texture(_array((4, 4, 4)), vg)
    assert tex.planes is not None
    s.reads_planes = 0
    K.set_params(params, pgs, vg)
    y = ([_array((5, 6), 0x900000 + 0x1000 * k) for k in range(3)] if as_list
         else _array((3, 5, 6)))
    K(tex, pgs, vg, y)          # (the pointer table is made once)
    del s.calls[:]
    for handle in (STREAM, None):
        K(tex, pgs, vg, y, stream=handle)
    build = "kk_volume_to_fp_texture"
    launch = "kk_cone_fp_ptrs" if as_list else "kk_cone_fp"
    assert s.of(build, launch) == [(build, STREAM), (launch, STREAM),
                                   (build, None), (launch, None)]


def test_new_pairs_wait_for_the_stream_they_are_allocated_on(stub):
    """Recycled memory is free on the current stream only: a launch on
    another stream that allocates the pairs waits for that one."""
    s = stub(1)
    tex = kernel.ProjectionTexture(3, 5, 6, like=_array((1,)))
    tex.update(_array((3, 5, 6)), planes=True)
    del s.calls[:]
    tex.pairs_ptr(STREAM)
    names = [c[0] for c in s.calls]
    assert names.index("kk_event_record") < names.index(
        "kk_stream_wait_event") < names.index("kk_projections_to_bp_texture")
    del s.calls[:]
    tex.pairs_ptr(STREAM)
    tex.pairs_ptr()
    assert s.of("kk_event_record", "kk_stream_wait_event") == []


def test_data_makes_the_pairs_the_content(stub):
    s = stub(1)
    for tex, src, build in (
            (kernel.ProjectionTexture(3, 5, 6, like=_array((1,))),
             _array((3, 5, 6)), "kk_projections_to_bp_texture"),
            (kernel.VolumeTexture((4, 4, 4), 0b001, like=_array((1,))),
             _array((4, 4, 4)), "kk_volume_to_fp_texture")):
        tex.update(src, planes=True)
        assert tex.planes is not None
        a = tex.ptr
        assert tex.planes is None and tex.ptr == a
        assert len(s.of(build)) == 1
