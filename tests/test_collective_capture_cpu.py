"""A decoding step with collectives is recorded in thread-local mode: while a recording is open under the global
mode, an event query of any other thread is an error, and the process group's watchdog thread queries the events of
the warm-up's collectives whenever it comes round to them.  The device calls are replaced by ones that do nothing."""
import types

import torch


def test_step_with_collectives_is_recorded_in_thread_local_mode(mv, monkeypatch):
    from micro_vllm_amd.core.layer.model_graph import ModelGraphRunner

    class Scope:
        def __init__(self, *a, **kw):
            modes.append(kw.get("capture_error_mode", "global")) if "stream" in kw else None

        def __enter__(self):
            return self

        def __exit__(self, *exc):
            return False

    modes, steps = [], []
    stream = types.SimpleNamespace(cuda_stream=4096, wait_stream=lambda other: None, synchronize=lambda: None)
    monkeypatch.setattr(torch.cuda, "Stream", lambda **kw: stream)
    monkeypatch.setattr(torch.cuda, "stream", Scope)
    monkeypatch.setattr(torch.cuda, "current_stream", lambda *a: stream)
    monkeypatch.setattr(torch.cuda, "CUDAGraph", lambda: "graph")
    monkeypatch.setattr(torch.cuda, "graph", Scope)
    runner = types.SimpleNamespace(device="cpu", _input_ids=torch.zeros(4, dtype=torch.long),
                                   decode=lambda ids, bs, cache: steps.append(bs))
    assert ModelGraphRunner._capture_one(runner, 4, None, 2, True) == "graph"
    assert steps == [4, 4, 4] and modes == ["thread_local"]
