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
        calls.append(step)
        return torch.empty_like(q)

    monkeypatch.setattr(attention.T, "prompt_layer", prompt_layer)
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


@pytest.mark.parametrize("lens,heads,kv_heads,step", [
    ([6] * 100, 32, 32, False), ([6] * 100, 64, 8, False), ([16] * 64, 52, 52, False), ([20] * 16, 52, 52, False),
    ([45] * 128, 32, 8, False), ([100] * 2, 64, 8, False), ([45], 32, 32, False), ([400], 32, 32, False),
    ([30] * 16, 32, 32, True), ([45] * 16, 32, 32, True), ([100] * 4, 64, 8, True), ([128] * 128, 32, 8, True),
    ([600], 32, 32, True), ([2048] * 4, 52, 52, True)])
def test_prompt_steps_take_the_faster_of_the_two_forms(monkeypatch, lens, heads, kv_heads, step):
    """Many short prompts keep rotation and cache write in a launch of their own
    (as part of the attention kernel they took up to 1.5 times as long), long ones
    and grouped queries do not."""
    assert _prompt_route(monkeypatch, lens, heads, kv_heads) is step
