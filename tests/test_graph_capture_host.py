"""Host side of ``Graph.capture``: what it does with Python's collector and
with library objects that die while a stream records, shown with a stub in the
library's place."""
import gc
import sys
import threading

import pytest

kk = pytest.importorskip("kernelkit")
from kernelkit import _native, device  # noqa: E402


class _StubLibrary:
    """Hands out handles, records calls; ``begin`` is begin_capture's
    status."""

    def __init__(self, begin=_native.KK_OK):
        self.begin = begin
        self.calls = []
        self._next = 1

    def __getattr__(self, name):
        if not name.startswith("kk_"):
            raise AttributeError(name)

        def call(*args):
            self.calls.append(name)
            if name == "kk_last_error":
                return b"stub"
            if name == "kk_graph_begin_capture":
                return self.begin
            if name.endswith("_create") or name in ("kk_malloc",
                                                    "kk_graph_end_capture"):
                out = args[1] if name == "kk_graph_end_capture" else args[0]
                out._obj.value = self._next
                self._next += 1
            return _native.KK_OK
        return call


@pytest.fixture
def stub(monkeypatch):
    def use(**kw):
        s = _StubLibrary(**kw)
        monkeypatch.setattr(_native, "lib", lambda: s)
        monkeypatch.setattr(_native, "_lib", s)
        return s
    yield use
    assert gc.isenabled()
    # no stub handle may reach the real library
    gc.collect()
    for o in gc.get_objects():
        if type(o) in (_native.Plan, _native.Batch, _native.Filter,
                       _native.Stream, _native.Event, _native.Graph):
            if o._ptr is not None and (o._ptr.value or 0) < 4096:
                o._ptr = None


def test_failed_begin_leaves_the_collector_alone(stub):
    stub(begin=_native.KK_ERR_HIP)
    try:
        with pytest.raises(_native.KernelError):
            _native.Graph.capture(lambda: None)
        assert gc.isenabled()
    finally:
        gc.enable()


def test_captures_of_two_threads_do_not_meet(stub):
    """The collector is as the program left it, in every thread, while
    captures of other threads begin and end."""
    stub()
    inside, over = threading.Event(), threading.Event()
    seen = []

    def first():
        inside.set()
        assert over.wait(30)
        seen.append(gc.isenabled())

    t = threading.Thread(target=_native.Graph.capture, args=(first,))
    t.start()
    assert inside.wait(30)
    try:
        seen.append(gc.isenabled())
        _native.Graph.capture(lambda: seen.append(gc.isenabled()))
        seen.append(gc.isenabled())
    finally:
        over.set()
        t.join()
    assert seen == [True] * 4


@pytest.mark.parametrize("fails", [False, True])
def test_objects_that_die_in_a_capture_are_freed_after_it(stub, fails):
    """A capture does not survive a free: what the collector (or the recorded
    function) drops meanwhile is freed once the capture has ended, also when
    the function raises."""
    s = stub()

    class Knot:
        pass

    frees = ("kk_plan_destroy", "kk_batch_destroy", "kk_filter_destroy",
             "kk_free", "kk_event_destroy", "kk_stream_destroy",
             "kk_graph_destroy")

    def body():
        for owner in (_native.Plan, _native.Batch, _native.Filter,
                      lambda: device._Buffer(64), _native.Event,
                      _native.Stream):
            k = Knot()
            k.self, k.owned = k, owner()
        old = _native.Graph(_native._vp(77))
        k.self = None
        del k, owner, old
        gc.collect()
        assert not set(frees) & set(s.calls)
        if fails:
            raise RuntimeError("from the body")

    if fails:
        with pytest.raises(RuntimeError, match="from the body"):
            _native.Graph.capture(body)
    else:
        g = _native.Graph.capture(body)
        del g
    gc.collect()
    end = s.calls.index("kk_graph_end_capture")
    for name in frees:
        assert name in s.calls[end:], name
        assert name not in s.calls[:end], name


def test_another_thread_frees_at_once(stub):
    s = stub()

    def body():
        t = threading.Thread(target=lambda: _native.Plan())
        t.start()
        t.join()
        assert "kk_plan_destroy" in s.calls

    _native.Graph.capture(body)


def test_a_capture_inside_a_capture_keeps_the_outer_ones_objects(stub):
    s = stub()

    def body():
        _native.Plan()
        _native.Graph.capture(lambda: None)
        assert "kk_plan_destroy" not in s.calls

    _native.Graph.capture(body)
    assert "kk_plan_destroy" in s.calls


def test_objects_that_outlive_the_module_say_nothing(stub, monkeypatch):
    """At the interpreter's end a module's names may be gone before the last
    objects are."""
    stub()
    owned = [_native.Plan(), _native.Batch(), _native.Filter(),
             _native.Stream(), _native.Event(), device._Buffer(4),
             _native.Graph(_native._vp(77))]
    said = []
    monkeypatch.setattr(sys, "unraisablehook", said.append)
    for name in ("release", "_local", "_lib", "lib", "_vp"):
        monkeypatch.setattr(_native, name, None)
    monkeypatch.setattr(device, "ctypes", None)
    monkeypatch.setattr(device, "_native", None)
    del owned
    gc.collect()
    assert said == []
