"""Kernels asked by several threads which layout they read, shown with a stub
in the library's place."""
import threading

import pytest

kk = pytest.importorskip("kernelkit")
from kernelkit import _native, workloads  # noqa: E402
from kernelkit.kernels.cone_bp import VoxelDrivenConeBP  # noqa: E402
from kernelkit.kernels.cone_fp import RayDrivenConeFP  # noqa: E402


class _StubLibrary:
    """``during(name)`` runs in the midst of each call."""

    def __init__(self):
        self.during = lambda name: None

    def __getattr__(self, name):
        if not name.startswith("kk_"):
            raise AttributeError(name)

        def call(*args):
            if name == "kk_plan_create":
                args[0]._obj.value = 0   # nothing to free
            self.during(name)
            if name.endswith("_reads_planes"):
                return 1
            if name == "kk_fp_frame_mask":
                return 0b011
            return _native.KK_OK
        return call


@pytest.fixture
def stub(monkeypatch):
    s = _StubLibrary()
    monkeypatch.setattr(_native, "lib", lambda: s)
    monkeypatch.setattr(_native, "_lib", s)
    return s


def _in_thread(fn):
    out = []
    t = threading.Thread(target=lambda: out.append(fn()))
    t.start()
    t.join()
    return out[0]


def _geometry():
    return (workloads.circular_geometry(3, 40.0, 20.0, 5, 6, 1.0),
            kk.resolve_volume_geometry(shape=(4, 4, 4), voxel_size=1.0))


def test_backprojection_answer_and_its_question_appear_together(stub):
    pgs, vg = _geometry()
    K = VoxelDrivenConeBP()
    K.compile()
    K.set_params(K.geoms2params(pgs, vg))
    seen = []

    def during(name):
        if name == "kk_bp_reads_planes" and not seen:
            seen.append(None)
            seen.append(_in_thread(lambda: K.reads_planes_for(5, 6, vg)))

    stub.during = during
    assert K.reads_planes_for(5, 6, vg) is True
    assert seen[1] is True and K.reads_planes


def test_forward_upload_is_seen_whole_or_not_at_all(stub):
    """A second thread sees the parameters as uploaded only once the frames
    and the layout that belong to them are known."""
    pgs, vg = _geometry()
    K = RayDrivenConeFP()
    K.compile()
    seen = []
    stub.during = lambda name: seen.append(
        _in_thread(lambda: (K.frame_mask, K.reads_planes))
        if name in ("kk_fp_frame_mask", "kk_fp_reads_planes") else (0, False))
    K.set_params(K.geoms2params(pgs, vg), pgs, vg)
    assert set(seen) == {(0, False)}
    assert (K.frame_mask, K.reads_planes) == (0b011, True)
