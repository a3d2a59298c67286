"""Workspaces whose addresses a recorded step replays: they live as long as the recording, and no other call gets them.

The device calls around a recording are replaced by ones that do nothing; the buffers are host tensors."""
import gc
import threading
import types
import weakref

import pytest
import torch


class _Stream:
    cuda_stream = 4096      # every stream has this handle: torch deals out 32 and starts again

    def wait_stream(self, other):
        pass

    def synchronize(self):
        pass


@pytest.fixture()
def nv(mv, monkeypatch):
    from micro_vllm_amd import _native

    class Scope:
        def __init__(self, stream):
            pass

        def __enter__(self):
            return self

        def __exit__(self, *exc):
            return False

    stream = _Stream()
    monkeypatch.setattr(torch.cuda, "Stream", lambda **kw: stream)
    monkeypatch.setattr(torch.cuda, "stream", Scope)
    monkeypatch.setattr(torch.cuda, "current_stream", lambda *a: stream)
    monkeypatch.setattr(_native, "_stream_ws", {})
    monkeypatch.setattr(_native, "lib", lambda: types.SimpleNamespace(
        mv_graph_begin_capture=lambda s: 0, mv_graph_end_capture=lambda s, h: 0, mv_graph_destroy=lambda h: 0))
    return _native


def _step(nv, sizes, handed, fail_at=None):
    """A runner's `_run` that asks for workspaces as its projections would."""
    runs = []

    def run(step, cache, want, residuals):
        runs.append(1)
        if fail_at == len(runs):
            raise RuntimeError("refused while recording")
        for n in sizes:
            handed.append(nv.stream_workspace("wgemm", "cpu:0", n))
        return torch.zeros(1)

    return types.SimpleNamespace(device="cpu", _run=run, _arena=None, _arena_off=0, _measured=0)


def _capture(runner, rows=2):
    from micro_vllm_amd.core.layer.ragged_runner import RaggedRunner

    return RaggedRunner._capture(runner, types.SimpleNamespace(rows=rows, slots=[0]), types.SimpleNamespace(states={}))


def test_a_recording_keeps_what_it_writes_to(nv):
    handed = []
    entry = _capture(_step(nv, [1000, 4000, 2000], handed))
    recorded = [weakref.ref(t) for t in handed[3:]]      # (the first three: the run that sizes things)
    assert len({t.data_ptr() for t in handed[3:]}) == 1 and handed[3].numel() * 4 >= 4000
    del handed[:]
    # a later recording of more rows, and the program's own calls, on a stream of the same handle
    later = []
    other = _capture(_step(nv, [9000], later), rows=32)
    grown = nv.stream_workspace("wgemm", "cpu:0", 20000)
    gc.collect()
    assert all(r() is not None for r in recorded)
    places = {recorded[0]().data_ptr(), later[-1].data_ptr(), grown.data_ptr()}
    assert len(places) == 3
    assert nv.stream_workspace("wgemm", "cpu:0", 100) is grown
    del entry
    gc.collect()
    assert recorded[0]() is None        # ... and no longer than it lives
    assert other


def test_calls_outside_a_recording_have_the_streams_own(nv):
    before = nv.stream_workspace("wgemm", "cpu:0", 100)
    with nv.own_workspaces() as table:
        inside = nv.stream_workspace("wgemm", "cpu:0", 50)
        assert inside is not before and list(table.values()) == [inside]
        seen = []
        t = threading.Thread(target=lambda: seen.append(nv.stream_workspace("wgemm", "cpu:0", 100)))
        t.start()
        t.join()
        assert seen[0] is before       # another thread's calls are not recorded
        with nv.own_workspaces():
            assert nv.stream_workspace("wgemm", "cpu:0", 50) is not inside
        assert nv.stream_workspace("wgemm", "cpu:0", 50) is inside
    assert nv.stream_workspace("wgemm", "cpu:0", 100) is before


@pytest.mark.parametrize("fail_at", [1, 2])
def test_a_recording_that_fails_leaves_nothing_behind(nv, fail_at):
    handed = []
    with pytest.raises(RuntimeError):
        _capture(_step(nv, [1000], handed, fail_at))
    assert nv._stream_ws == {}
    assert nv.stream_workspace("wgemm", "cpu:0", 10) is nv._stream_ws[("wgemm", 0, _Stream.cuda_stream)]
