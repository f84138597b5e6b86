"""Which operator a step of PagedAttentionWithRoPE takes (no GPU: the operators are
replaced by recorders)."""
import pytest
import torch

from muxserve_amd import attention
from muxserve_amd.attention import InputMetadata, PagedAttentionWithRoPE

D = attention.HEAD_SIZE


def _prompt_route(monkeypatch, lens, heads, kv_heads):
    calls = []

    def prompt_layer(positions, q, k, v, cos_sin, k_pool, v_pool, slots, layer, cu_seqlens, prompt_lens, scale, step):
        calls.append("step" if step else "one launch")
        return torch.empty_like(q)

    monkeypatch.setattr(attention.T, "prompt_layer", prompt_layer)
    monkeypatch.setattr(attention.T, "rotary_neox", lambda *a, **kw: calls.append("two launches"))
    for name in ("reshape_and_cache", "prefill_causal"):
        monkeypatch.setattr(attention.T, name, lambda *a, **kw: None)
    n = sum(lens)
    none = torch.empty((0,), dtype=torch.int32)
    md = InputMetadata(prompt_lens=lens, slot_mapping=torch.zeros((n, 1, kv_heads), dtype=torch.int64), context_lens=none,
                       max_context_len=0, block_tables=none.view(0, 0, 0, 0))
    layer = PagedAttentionWithRoPE(heads, D, D ** -0.5, max_position=64, rotary_dim=D, num_kv_heads=kv_heads)
    q = torch.empty((n, heads * D), dtype=torch.float16)
    k, v = (torch.empty((n, kv_heads * D), dtype=torch.float16) for _ in range(2))
    layer(torch.zeros(n, dtype=torch.int64), q, k, v, torch.empty(0), torch.empty(0), md, None)
    assert len(calls) == 1
    return calls[0]


@pytest.mark.parametrize("lens,heads,kv_heads,route", [
    ([6] * 100, 32, 32, "one launch"), ([6] * 100, 64, 8, "two launches"), ([13] * 40, 64, 8, "two launches"),
    ([45] * 16, 16, 2, "one launch"),
    ([16] * 64, 52, 52, "one launch"), ([20] * 16, 52, 52, "one launch"), ([45] * 128, 32, 8, "two launches"),
    ([100] * 2, 64, 8, "one launch"), ([45], 32, 32, "one launch"), ([400], 32, 32, "one launch"),
    ([30] * 16, 32, 32, "step"), ([45] * 16, 32, 32, "step"), ([100] * 4, 64, 8, "step"), ([128] * 128, 32, 8, "step"),
    ([600], 32, 32, "step"), ([2048] * 4, 52, 52, "step")])
def test_prompt_steps_take_the_faster_form(monkeypatch, lens, heads, kv_heads, route):
    """Many short prompts keep rotation and cache write out of the attention kernel
    (as part of it they took up to 1.5 times as long), long ones do not."""
    assert _prompt_route(monkeypatch, lens, heads, kv_heads) == route


def test_decode_layer_does_without_torchs_private_stream_handle(monkeypatch):
    """The workspace of the decode operator is looked up under the current stream's
    handle, with or without torch's private function for it."""
    from types import SimpleNamespace
    from muxserve_amd import ops, torch_ops
    device, ws, seen = torch.device("cuda", 0), object(), []

    def op(*args):
        seen.append(args[-2])
        return "out", 0

    monkeypatch.setattr(torch_ops, "load", lambda: SimpleNamespace(decode_layer=op))
    monkeypatch.setattr(torch.cuda, "current_stream", lambda d: SimpleNamespace(cuda_stream=7))
    monkeypatch.setitem(ops._workspaces, (device, 7), ws)
    q = SimpleNamespace(device=device)
    for raw in (None, lambda index: 7):
        monkeypatch.setattr(torch_ops, "_raw_stream", raw, raising=False)
        assert torch_ops.decode_layer(None, q, *[None] * 14) == "out"
    assert seen == [ws, ws]
