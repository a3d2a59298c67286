"""What the Llama-shaped prefill refuses before its one native call is made (no GPU: the library is a stand-in that must
not be reached)."""
from types import SimpleNamespace

import pytest
import torch


def _runner(monkeypatch, on_gpu=lambda t: True):
    from micro_vllm_amd.core.layer import model_prefill as mp

    class Lib:
        def mv_llama_prefill_workspace_bytes(self, *a):
            return 0

        def mv_llama_prefill_layers(self, *a):
            raise RuntimeError("launched")

    monkeypatch.setattr(mp.nv, "lib", lambda: Lib())
    monkeypatch.setattr(mp.nv, "stream_ptr", lambda: 0)
    monkeypatch.setattr(torch.Tensor, "is_cuda", property(on_gpu))
    hid, hq, hkv, d, inter = 64, 2, 1, 32, 128
    W = lambda n, k, swiglu=False: SimpleNamespace(tiles=torch.zeros(1), n=n, k=k, swiglu=swiglu,   # noqa: E731
                                                   out_features=n // 2 if swiglu else n)
    norm = lambda: SimpleNamespace(weight=torch.ones(hid, dtype=torch.bfloat16), eps=1e-5)          # noqa: E731
    blocks = [SimpleNamespace(ln_1=norm(), ln_2=norm(), attn=SimpleNamespace(_qkv_w=W((hq + 2 * hkv) * d, hid), _qkv_b=None,
                                                                             _o=W(hid, hq * d)),
                              mlp=SimpleNamespace(_gu=W(2 * inter, hid, True), _d=W(hid, inter))) for _ in range(2)]
    r = mp.ModelPrefillRunner.__new__(mp.ModelPrefillRunner)
    r.hidden_dim, r.num_heads, r.kv_num_heads, r.head_size, r.num_layers = hid, hq, hkv, d, 2
    r.model = SimpleNamespace(transformer=SimpleNamespace(h=blocks))
    table = torch.ones(16, d // 2, dtype=torch.bfloat16)
    r.attention = SimpleNamespace(_cos_pool=table, _sin_pool=table)
    kv = torch.zeros(3, 64, hkv, d, dtype=torch.bfloat16)
    return r, SimpleNamespace(get=lambda li: (kv, kv)), torch.zeros(2 * 5, hid, dtype=torch.bfloat16)


def _call(r, mgr, h, lens=2, rows=2):
    return r._prefill_stack(h, 2, 5, mgr, torch.zeros(lens, dtype=torch.int32), torch.zeros(rows, 4, dtype=torch.int32))


def test_well_formed_layers_are_launched(mv, monkeypatch):
    r, mgr, h = _runner(monkeypatch)
    with pytest.raises(RuntimeError, match="launched"):
        _call(r, mgr, h)


@pytest.mark.parametrize("lens,rows", [(1, 2), (2, 1)])
def test_more_rows_than_the_cache_managers_buffers_hold(mv, monkeypatch, lens, rows):
    """A batch above the manager's max_batch_size leaves its slices short; reading on would leave the buffers."""
    r, mgr, h = _runner(monkeypatch)
    with pytest.raises(AssertionError):
        _call(r, mgr, h, lens, rows)


def test_norm_weights_in_host_memory(mv, monkeypatch):
    held = []
    r, mgr, h = _runner(monkeypatch, on_gpu=lambda t: not any(t is x for x in held))
    held.append(r.model.transformer.h[1].ln_2.weight)
    with pytest.raises(AssertionError):
        _call(r, mgr, h)


def test_rotary_tables_of_another_head_size(mv, monkeypatch):
    r, mgr, h = _runner(monkeypatch)
    r.attention._cos_pool = torch.ones(16, 8, dtype=torch.bfloat16)
    with pytest.raises(AssertionError):
        _call(r, mgr, h)


def test_an_empty_batch_needs_no_launch(mv, monkeypatch):
    r, mgr, h = _runner(monkeypatch)
    out = r._prefill_stack(h[:0], 2, 0, mgr, torch.zeros(2, dtype=torch.int32), torch.zeros(2, 4, dtype=torch.int32))
    assert out is not None and out.shape[0] == 0
