"""The drop-in boundary end to end on the GPU: two models of different head and
layer counts share ONE pool and ONE KVStorage; every step goes
BatchScheduler -> allocator -> prepare_inputs -> PagedAttentionWithRoPE.forward
for every layer, exactly as the reference's serving loop drives its attention
layer (llm_runtime.py:277-339, models/llama.py:149-163).  Checked per layer
against the oracle; the pool is compared bit-exact at the end.
"""
import ctypes
import os
import re

import numpy as np
import pytest
import torch

from oracle import attn_oracle as orc
from muxserve_amd import ops
from muxserve_amd.attention import PagedAttentionWithRoPE
from muxserve_amd.batch_scheduler import BatchScheduler
from muxserve_amd.device_tables import DeviceBlockTables
from muxserve_amd.memory_manager import KVStorage
from muxserve_amd.pool import HEAD_SIZE, allocate_gpu_cache
from muxserve_amd.prepare import prepare_inputs

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
D = HEAD_SIZE
TOL = 2e-3


class _Model:
    def __init__(self, name, L, Hq, Hkv, storage, bs, seed, fused_rope_max_tokens=512, device_rows=0):
        self.name, self.L, self.Hq, self.Hkv = name, L, Hq, Hkv
        self.sched = BatchScheduler(L, Hkv, 512, bs)
        self.storage = storage
        self.layers = [PagedAttentionWithRoPE(Hq, D, D ** -0.5, base=10000, max_position=2048, rotary_dim=D,
                                              num_kv_heads=Hkv, rope_scaling=None, layer_idx=l) for l in range(L)]
        for layer in self.layers:
            layer.fused_rope_max_tokens = fused_rope_max_tokens
        self.g = torch.Generator().manual_seed(seed)
        self.device_tables = DeviceBlockTables(self.sched, device_rows, DEV) if device_rows else None

    def alloc(self, req):
        return self.storage.allocate_batch(req, self.L, self.Hkv)


def _step(m, ids, last_tokens, k_pool, v_pool, hk, hv, permuted):
    tokens, positions, md, batch_reqs, preempted = prepare_inputs(m.sched, m.alloc, ids, last_tokens, DEV,
                                                                  permuted_tables=permuted,
                                                                  device_tables=m.device_tables)
    assert not preempted
    T_pad = tokens.shape[0]
    n = md.num_valid_tokens
    worst = 0.0
    for l, layer in enumerate(m.layers):
        qkv = torch.randn((T_pad, (m.Hq + 2 * m.Hkv) * D), generator=m.g).half()
        dqkv = qkv.to(DEV)
        q, k, v = dqkv.split([m.Hq * D, m.Hkv * D, m.Hkv * D], dim=-1)          # models/llama.py:157-158
        q0, k0 = qkv[:, :m.Hq * D].clone(), qkv[:, m.Hq * D:(m.Hq + m.Hkv) * D].clone()
        out = layer(positions, q, k, v, k_pool, v_pool, md, None)
        torch.cuda.synchronize()
        # rotary: in place on q and k, against the textbook form (one fp16 rounding apart)
        rq, rk = orc.rotary_neox(positions[:n].cpu(), q0, k0)
        gq, gk = q[:n].cpu(), k[:n].cpu()
        assert (gq.float() - rq).abs().max() <= 4e-3 and (gk.float() - rk).abs().max() <= 4e-3
        assert torch.equal(q[n:].cpu(), q0[n:]) and torch.equal(k[n:].cpu(), k0[n:]), "padding rows rotated"
        # cache write + attention: the oracle consumes the GPU's rotated q, k so
        # that the comparison isolates the scatter (bit-exact) and the attention
        hv_in = qkv[:, (m.Hq + m.Hkv) * D:]
        orc.reshape_and_cache(gk, hv_in, hk, hv, md.slot_mapping.cpu(), layer=l, num_tokens=n)
        if md.num_prompt_tokens:
            want = orc.prefill_causal(gq, gk, hv_in[:n], md.prompt_lens, D ** -0.5, m.Hkv)
        else:
            want = orc.paged_decode(gq, hk, hv, md.block_tables.cpu(), md.context_lens.cpu().numpy(), D ** -0.5,
                                    layer=l)
        err = (out[:n].float().cpu() - want).abs().max().item()
        assert err <= TOL, f"{m.name} layer {l}: max-abs error {err:.3e}"
        worst = max(worst, err)
    return worst


@pytest.mark.parametrize("permuted,fused_max,device_rows", [(True, 512, 0), (False, 512, 0), (True, 0, 0),
                                                            (True, 60, 0), (True, 512, 8)])
def test_two_models_share_one_pool_prefill_then_decode(permuted, fused_max, device_rows):
    """fused_max: steps of up to that many tokens rotate and write the cache in
    one launch (0: always the two kernels; 60: decode steps fused, prefill not).
    device_rows > 0: slot mapping and block tables are built on the device."""
    print(f"[case] serving path permuted_tables={permuted} fused_rope_max_tokens={fused_max} "
          f"device_rows={device_rows}", flush=True)
    bs, N = 16, 6000
    storage = KVStorage(N)
    k_pool, v_pool = allocate_gpu_cache(N, bs, DEV)
    k_pool.zero_()
    v_pool.zero_()
    hk, hv = k_pool.cpu(), v_pool.cpu()
    a = _Model("small-mha", 2, 4, 4, storage, bs, seed=1, fused_rope_max_tokens=fused_max, device_rows=device_rows)
    b = _Model("gqa", 3, 8, 2, storage, bs, seed=2, fused_rope_max_tokens=fused_max, device_rows=device_rows)
    rng = np.random.Generator(np.random.PCG64(3))
    for m, lens, base_id in ((a, [5, 40, 17], 0), (b, [130, 16, 1, 33], 100)):
        for i, p in enumerate(lens):
            m.sched.add_request(rng.integers(0, 24000, size=p).astype(np.int32), base_id + i, 64)
    ids_a, ids_b = [0, 1, 2], [100, 101, 102, 103]
    _step(a, ids_a, [], k_pool, v_pool, hk, hv, permuted)           # prefill, model a
    _step(b, ids_b, [], k_pool, v_pool, hk, hv, permuted)           # prefill, model b (interleaved blocks)
    for step in range(20):                                          # decode, crossing block boundaries
        _step(a, ids_a, [7 + step] * 3, k_pool, v_pool, hk, hv, permuted)
        _step(b, ids_b[::-1], [9 + step] * 4, k_pool, v_pool, hk, hv, permuted)
    # one model's sequence finishes; its blocks are reused by a new request of the other model
    storage.free_batch([1])
    a.sched.release_requests([1])
    b.sched.add_request(rng.integers(0, 24000, size=70).astype(np.int32), 104, 64)
    _step(b, [104], [], k_pool, v_pool, hk, hv, permuted)
    for step in range(3):
        _step(a, [0, 2], [1, 2], k_pool, v_pool, hk, hv, permuted)
        _step(b, ids_b + [104], [3] * 5, k_pool, v_pool, hk, hv, permuted)
    assert torch.equal(k_pool.cpu().view(torch.int16), hk.view(torch.int16))
    assert torch.equal(v_pool.cpu().view(torch.int16), hv.view(torch.int16))
    assert storage.num_free() + sum(storage.num_held(i) for i in [0, 2, 100, 101, 102, 103, 104]) == N


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("Hq,Hkv", [(3, 3), (8, 2)])
@pytest.mark.parametrize("bs", [16, 8])
def test_fused_rotary_cache_write_equals_the_two_kernels(dtype, Hq, Hkv, bs):
    """mux_rope_reshape_and_cache against mux_rotary_neox followed by
    mux_reshape_and_cache on the same inputs: q, k and both pools bitwise equal.
    Packed ragged prompts (runs at every phase) plus tokens without a slot,
    which are rotated but not written."""
    print(f"[case] fused rope + cache write {dtype} Hq={Hq} Hkv={Hkv} bs={bs}", flush=True)
    from muxserve_amd import workloads
    from muxserve_amd.attention import build_cos_sin_cache
    from muxserve_amd.pool import allocate_gpu_cache
    rng = np.random.Generator(np.random.PCG64(77 + bs))
    g = torch.Generator().manual_seed(77 + bs)
    lens = rng.permutation(np.arange(1, 30)).astype(np.int32)
    T = int(lens.sum())
    N = int(((lens + bs - 1) // bs).sum()) * Hkv + 5
    slots, _ = workloads.prefill_slot_mapping(lens, Hkv, bs, rng.permutation(N))
    slots[5, 0, 0] = -1
    slots[T - 1, 0, :] = -1
    pad = (T + 7) // 8 * 8
    qkv = torch.randn((pad, (Hq + 2 * Hkv) * D), generator=g).to(dtype).to(DEV)
    positions = torch.from_numpy(rng.integers(0, 2048, size=pad)).to(DEV)
    cos_sin = build_cos_sin_cache(D, 2048, 10000.0, DEV)
    dslots = torch.from_numpy(slots).to(DEV)
    results = []
    for fused in (False, True):
        x = qkv.clone()
        q, k, v = x.split([Hq * D, Hkv * D, Hkv * D], dim=-1)
        kp, vp = allocate_gpu_cache(N, bs, DEV, dtype=dtype)
        kp.zero_()
        vp.zero_()
        if fused:
            ops.rope_reshape_and_cache(positions, q, k, v, cos_sin, kp, vp, dslots, num_tokens=T)
        else:
            ops.rotary_neox(positions, q, k, cos_sin, num_tokens=T)
            ops.reshape_and_cache(k, v, kp, vp, dslots, num_tokens=T)
        torch.cuda.synchronize()
        results.append((x.cpu().view(torch.int16), kp.cpu().view(torch.int16), vp.cpu().view(torch.int16)))
    for a, b, what in zip(results[0], results[1], ("qkv rows", "k pool", "v pool")):
        assert torch.equal(a, b), f"{what} differ between the fused launch and the two kernels"
    assert torch.equal(results[1][0][T:], qkv.cpu().view(torch.int16)[T:]), "padding rows must not be touched"


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("bs", [16, 8, 32])
@pytest.mark.parametrize("T,Hq,Hkv", [(1, 1, 1), (9, 5, 5), (320, 16, 8), (321, 16, 8)])
def test_rotary_cache_write_on_both_sides_of_the_scatter_rule(dtype, bs, T, Hq, Hkv):
    """Steps of few (token, kv head) pairs take a kernel of their own (up to 2560
    = 320 x 8): one model and two models per call against rotary and cache write in
    turn, q, k and both pools bitwise equal.  Scattered slots, as decode steps
    have them, next to runs, missing slots and slots outside the pool."""
    print(f"[case] rotary + cache write {dtype} T={T} Hq={Hq} Hkv={Hkv} bs={bs}", flush=True)
    from muxserve_amd.attention import build_cos_sin_cache
    rng = np.random.Generator(np.random.PCG64(T + bs))
    g = torch.Generator().manual_seed(T + bs)
    N = 2 * (2 * T * Hkv // bs + 4)
    free = rng.permutation(N // 2 * bs)                                # model 0: anywhere in the first half
    slots = [free[:T * Hkv].reshape(T, 1, Hkv), (N // 2 * bs + np.arange(T * Hkv)).reshape(Hkv, T).T.reshape(T, 1, Hkv)]
    slots = [np.ascontiguousarray(s.astype(np.int64)) for s in slots]
    slots[0][T // 2, 0, 0] = -1
    slots[1][T - 1, 0, -1] = N * bs
    dslots = [torch.from_numpy(s).to(DEV) for s in slots]
    rows = [torch.randn((T, (Hq + 2 * Hkv) * D), generator=g).to(dtype).to(DEV) for _ in range(2)]
    positions = [torch.from_numpy(rng.integers(-2, 2050, size=T)).to(DEV) for _ in range(2)]
    cos_sin = build_cos_sin_cache(D, 2048, 10000.0, DEV)
    results = []
    for how in ("kernels", "one", "two"):
        xs = [x.clone() for x in rows]
        qkv = [x.split([Hq * D, Hkv * D, Hkv * D], dim=-1) for x in xs]
        kp, vp = allocate_gpu_cache(N, bs, DEV, dtype=dtype)
        kp.fill_(3)
        vp.fill_(5)
        if how == "two":
            ops.multi_reshape_and_cache([ops.CacheWriteCall(k, v, s, 0, p, cos_sin, q, T)
                                         for (q, k, v), s, p in zip(qkv, dslots, positions)], kp, vp)
        else:
            for (q, k, v), s, p in zip(qkv, dslots, positions):
                if how == "one":
                    ops.rope_reshape_and_cache(p, q, k, v, cos_sin, kp, vp, s)
                else:
                    ops.rotary_neox(p, q, k, cos_sin)
                    ops.reshape_and_cache(k, v, kp, vp, s)
        torch.cuda.synchronize()
        results.append([t.cpu().view(torch.int16) for t in (*xs, kp, vp)])
    for got in results[1:]:
        for a, b, what in zip(results[0], got, ("rows of model 0", "rows of model 1", "k pool", "v pool")):
            assert torch.equal(a, b), f"{what} differ from rotary and cache write in turn"


def _cache_write_line(name):
    """A limit of cache_write.hip's choice of kernels, from its source."""
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    text = open(os.path.join(root, "muxserve_amd", "csrc", "hip", "cache_write.hip")).read()
    return int(re.search(rf"constexpr int64_t {name} = (\d+);", text).group(1))


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("bs", [8, 16, 32])
@pytest.mark.parametrize("T,Hq,Hkv,kernel", [(435, 3, 3, "scatter"), (435, 5, 5, "scatter"), (2, 1, 1, "scatter"),
                                             (49, 52, 52, "scatter"), (64, 40, 40, "scatter"), (320, 32, 8, "scatter"),
                                             (65, 40, 40, "window"), (435, 8, 8, "window"),
                                             (435, 16, 8, "window"), (5119, 8, 8, "window"), (32767, 8, 8, "window"),
                                             (32768, 8, 8, "early"), (6560, 40, 40, "early"), (32769, 16, 8, "window")])
def test_rotary_cache_write_of_packed_prompts_in_each_kernel(dtype, bs, T, Hq, Hkv, kernel):
    """Packed ragged prompts (windows of up to 31 tokens, runs at every phase) in
    every form of the rotary cache write, as one call of one model and as one call
    of two models that hold the two halves of the tokens: rows and pools bitwise
    those of rotary and cache write in turn."""
    print(f"[case] packed prompts {dtype} bs={bs} T={T} Hq={Hq} Hkv={Hkv} {kernel}", flush=True)
    from muxserve_amd import workloads
    from muxserve_amd.attention import build_cos_sin_cache
    pairs, small, early = T * Hkv, _cache_write_line("kScatterPairs"), _cache_write_line("kEarlyQPairs")
    assert kernel == ("scatter" if pairs <= small else "early" if Hq == Hkv and pairs >= early else "window")
    rng = np.random.Generator(np.random.PCG64(T + bs))
    g = torch.Generator().manual_seed(T + bs)
    lens = []
    while sum(lens) < T:
        lens.append(min(int(rng.integers(1, min(60, T))), T - sum(lens)))
    half = len(lens) // 2
    N = sum((n + bs - 1) // bs for n in lens) * Hkv + 5
    slots, _ = workloads.prefill_slot_mapping(np.array(lens, dtype=np.int32), Hkv, bs, rng.permutation(N))
    slots[min(7, T - 1), 0, 0] = -1
    slots[T - 1, 0, :] = -1
    slots[T // 2, 0, -1] = N * bs
    dslots = torch.from_numpy(slots).to(DEV)
    qkv = torch.randn((T, (Hq + 2 * Hkv) * D), generator=g).to(dtype).to(DEV)
    positions = torch.from_numpy(rng.integers(-2, 2050, size=T)).to(DEV)
    cos_sin = build_cos_sin_cache(D, 2048, 10000.0, DEV)
    results = []
    for how in ("kernels", "one", "two"):
        x = qkv.clone()
        q, k, v = x.split([Hq * D, Hkv * D, Hkv * D], dim=-1)
        kp, vp = allocate_gpu_cache(N, bs, DEV, dtype=dtype)
        kp.fill_(3)
        vp.fill_(5)
        if how == "kernels":
            ops.rotary_neox(positions, q, k, cos_sin)
            ops.reshape_and_cache(k, v, kp, vp, dslots)
        elif how == "one":
            ops.rope_reshape_and_cache(positions, q, k, v, cos_sin, kp, vp, dslots)
        else:
            cut = sum(lens[:half])
            ops.multi_reshape_and_cache([ops.CacheWriteCall(k[a:b], v[a:b], dslots[a:b], 0, positions[a:b], cos_sin, q[a:b],
                                                            b - a) for a, b in ((0, cut), (cut, T))], kp, vp)
        results.append([t.view(torch.int16) for t in (x, kp, vp)])
    for got in results[1:]:
        for a, b, what in zip(results[0], got, ("qkv rows", "k pool", "v pool")):
            assert torch.equal(a, b), f"{what} differ from rotary and cache write in turn"


@pytest.mark.parametrize("bs", [8, 16, 32])
@pytest.mark.parametrize("T,H,rope", [(37, 3, True), (37, 3, False), (1100, 3, True), (1100, 3, False)])
def test_cache_write_of_tokens_by_themselves_and_in_runs(bs, T, H, rope):
    """Tokens without a neighbour in the slots beside theirs go past the L2, in both
    rotary kernels (2560 pairs apart) and the plain one: single tokens, pairs, runs of 3, 7,
    8, 9 and 16 from any offset, skipped tokens between them and slot 0, against a scatter
    in torch; slots that nobody writes keep their contents."""
    print(f"[case] cache write alone and in runs bs={bs} T={T} rope={rope}", flush=True)
    from muxserve_amd.attention import build_cos_sin_cache
    rng = np.random.Generator(np.random.PCG64(T + bs))
    N = 4 * T * H // bs + 8
    slots = np.full((T, 1, H), -1, dtype=np.int64)
    for h in range(H):
        lo, t = h * (N * bs // H), 0
        while t < T:
            n = min(int(rng.choice([1, 1, 1, 2, 3, 7, 8, 9, 16])), T - t)
            slots[t:t + n, 0, h] = lo + np.arange(n)
            lo += n + int(rng.integers(1, 4))
            t += n + int(rng.random() < 0.2)
    pad = (T + 7) // 8 * 8
    g = torch.Generator().manual_seed(T)
    x = torch.randn((pad, 3 * H * D), generator=g).half().to(DEV)
    q, k, v = x.split([H * D] * 3, dim=-1)
    positions = torch.arange(pad, device=DEV)
    kp, vp = allocate_gpu_cache(N, bs, DEV, dtype=torch.float16)
    kp.fill_(3)
    vp.fill_(5)
    dslots = torch.from_numpy(slots).to(DEV)
    if rope:
        ops.rope_reshape_and_cache(positions, q, k, v, build_cos_sin_cache(D, 2048, 10000.0, DEV), kp, vp, dslots, layer=0,
                                   num_tokens=T)
    else:
        ops.reshape_and_cache(k, v, kp, vp, dslots, layer=0, num_tokens=T)
    torch.cuda.synchronize()
    wk, wv = torch.full_like(kp, 3), torch.full_like(vp, 5)
    for h in range(H):
        sl = dslots[:, 0, h]
        ok = sl >= 0
        blk, off = sl[ok] // bs, sl[ok] % bs
        wk[blk, :, off, :] = k[:T, h * D:(h + 1) * D][ok].reshape(-1, D // 8, 8)       # (k as rotated in place)
        wv[blk, :, off] = v[:T, h * D:(h + 1) * D][ok]
    assert torch.equal(kp.view(torch.int16), wk.view(torch.int16)) and torch.equal(vp.view(torch.int16), wv.view(torch.int16))


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("Hq,Hkv,bs,many", [(3, 3, 16, False), (8, 2, 8, False), (16, 2, 32, False), (2, 1, 16, True)])
def test_prompt_step_operator_equals_the_three_kernels(dtype, Hq, Hkv, bs, many):
    """rope_prefill_and_cache against rotary, cache write and attention in turn:
    q, k, both pools and the outputs bitwise equal.  Prompt lengths around the
    tile and run sizes (or more prompts than the kernel argument lists), tokens
    without a slot, with a slot outside the pool, and a prompt whose slots are
    scattered token by token."""
    print(f"[case] prompt step operator {dtype} Hq={Hq} Hkv={Hkv} bs={bs} many={many}", flush=True)
    from muxserve_amd import torch_ops, workloads
    from muxserve_amd.attention import build_cos_sin_cache
    rng = np.random.Generator(np.random.PCG64(5 + bs))
    g = torch.Generator().manual_seed(5 + bs)
    lens = [1] * 400 + [2] * 400 if many else [1, 7, 8, 31, 32, 33, 127, 0, 128, 129, 257, 300]
    T, L, layer = sum(lens), 2, 1
    N = sum((n + bs - 1) // bs for n in lens) * Hkv + 5
    slots, _ = workloads.prefill_slot_mapping(np.array(lens, dtype=np.int32), Hkv, bs, rng.permutation(N))
    first = T - lens[-1]
    slots[first:, 0, :] = slots[first + rng.permutation(lens[-1]), 0, :]
    slots[first + 40:first + 56, 0, :] = np.sort(slots[first + 40:first + 56, 0, :], axis=0)
    slots[T // 2, 0, 0] = -1
    slots[T - 1, 0, :] = -1
    slots[T // 3, 0, -1] = N * bs
    slots = np.concatenate([np.full_like(slots, -1), slots], axis=1)        # layer 1 of 2
    pad = (T + 7) // 8 * 8
    qkv = torch.randn((pad, (Hq + 2 * Hkv) * D), generator=g).to(dtype).to(DEV)
    positions = torch.from_numpy(rng.integers(-3, 2060, size=pad)).to(DEV)   # clamped to the table
    cos_sin = build_cos_sin_cache(D, 2048, 10000.0, DEV)
    dslots = torch.from_numpy(slots).to(DEV)
    cu = torch.tensor(np.concatenate([[0], np.cumsum(lens)]), dtype=torch.int32, device=DEV)
    results = []
    for fused in (False, True):
        x = qkv.clone()
        q, k, v = x.split([Hq * D, Hkv * D, Hkv * D], dim=-1)
        kp, vp = allocate_gpu_cache(N, bs, DEV, dtype=dtype)
        kp.fill_(3)
        vp.fill_(5)
        out = torch.zeros((pad, Hq * D), dtype=dtype, device=DEV)
        if fused:
            torch_ops.rope_prefill_and_cache(out, positions, q, k, v, cos_sin, kp, vp, dslots, layer, cu, lens, D ** -0.5)
        else:
            ops.rotary_neox(positions, q, k, cos_sin, num_tokens=T)
            ops.reshape_and_cache(k, v, kp, vp, dslots, layer=layer, num_tokens=T)
            ops.prefill_causal(out[:T], q[:T], k[:T], v[:T], cu, max(lens), D ** -0.5, Hkv, prompt_lens=lens)
        torch.cuda.synchronize()
        results.append([t.cpu().view(torch.int16) for t in (x, kp, vp, out)])
    for a, b, what in zip(*results, ("qkv rows", "k pool", "v pool", "outputs")):
        assert torch.equal(a, b), f"{what} differ between the step operator and the three kernels"


def _captured_launches(fn):
    """Threads per workgroup of every kernel that fn launches, in order, from a graph of it
    (which is not run; fn runs once before, for its workspaces on that stream)."""
    hip = ctypes.CDLL(next(line.split()[-1] for line in open("/proc/self/maps") if "libamdhip64" in line))

    class Params(ctypes.Structure):                  # hipKernelNodeParams
        _fields_ = [("block", ctypes.c_uint32 * 3), ("extra", ctypes.c_void_p), ("func", ctypes.c_void_p),
                    ("grid", ctypes.c_uint32 * 3), ("params", ctypes.c_void_p), ("shared", ctypes.c_uint32)]

    stream, captured = torch.cuda.Stream(), torch.cuda.CUDAGraph(keep_graph=True)
    torch.cuda.synchronize()
    with torch.cuda.stream(stream):
        fn()
    stream.synchronize()
    with torch.cuda.graph(captured, stream=stream):
        fn()
    graph, n = ctypes.c_void_p(captured.raw_cuda_graph()), ctypes.c_size_t()
    assert hip.hipGraphGetNodes(graph, None, ctypes.byref(n)) == 0
    nodes = (ctypes.c_void_p * n.value)()
    assert hip.hipGraphGetNodes(graph, nodes, ctypes.byref(n)) == 0
    threads = []
    for node in nodes:
        kind, params = ctypes.c_int(), Params()
        assert hip.hipGraphNodeGetType(ctypes.c_void_p(node), ctypes.byref(kind)) == 0 and kind.value == 0
        assert hip.hipGraphKernelNodeGetParams(ctypes.c_void_p(node), ctypes.byref(params)) == 0
        threads.append(params.block[0])
    return threads


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("lens,H,bs,waves", [
    ([1, 7, 16, 17, 32, 33, 0, 127, 128], 3, 16, 4), ([45], 2, 8, 4), ([30, 5], 4, 16, 4),                 # few
    ([1, 7, 16, 17, 32, 33, 0, 127, 128] * 4, 8, 16, 4), ([128, 65, 100, 97, 31, 127] * 7, 8, 32, 4),
    ([1, 2, 15, 16, 17, 31, 32, 0] * 12, 8, 16, 1), ([1] * 220 + [9] * 7, 7, 32, 1), ([1] * 520 + [9] * 7, 1, 32, 0),  # many
    ([1, 3, 17, 32] * 200, 1, 16, 1),                                  # (more than a launch lists one by one)
    ([33, 64, 48, 63, 16, 1, 40] * 10, 8, 16, 2), ([64, 17, 47] * 30, 7, 8, 2), ([64, 1, 1, 1, 1] * 12, 10, 16, 0),
    ([128, 65, 100, 97, 31, 127] * 12, 8, 32, 4), ([96, 113, 128] * 30, 6, 16, 4), ([128, 3, 1] * 30, 6, 16, 0)])
def test_short_prompts_in_one_launch_equal_the_three_kernels(dtype, lens, H, bs, waves):
    """Steps of prompts of at most 128 tokens (one launch of workgroups of 1, 2 or 4
    waves, as stated; 0: two launches): q, k, both pools and the outputs bitwise as from
    rotary, cache write and attention in turn; with tokens without a slot, one outside the
    pool and a prompt whose slots are scattered token by token."""
    print(f"[case] short prompts {dtype} {len(lens)} prompts up to {max(lens)} H={H} bs={bs}", flush=True)
    from muxserve_amd import torch_ops, workloads
    from muxserve_amd.attention import build_cos_sin_cache
    rng = np.random.Generator(np.random.PCG64(len(lens) + bs))
    T = sum(lens)
    N = sum((n + bs - 1) // bs for n in lens) * H + 3
    slots, _ = workloads.prefill_slot_mapping(np.array(lens, dtype=np.int32), H, bs, rng.permutation(N))
    first = T - lens[-1]
    slots[first:, 0, 0] = slots[first + rng.permutation(lens[-1]), 0, 0]
    slots[T // 2, 0, 0] = -1
    slots[T // 3, 0, -1] = N * bs
    dslots = torch.from_numpy(slots).to(DEV)
    pad = (T + 7) // 8 * 8
    qkv = torch.randn((pad, 3 * H * D), generator=torch.Generator().manual_seed(T)).to(dtype).to(DEV)
    positions = torch.from_numpy(rng.integers(-3, 2060, size=pad)).to(DEV)
    cos_sin = build_cos_sin_cache(D, 2048, 10000.0, DEV)
    cu = torch.tensor(np.concatenate([[0], np.cumsum(lens)]), dtype=torch.int32, device=DEV)
    results = []
    for fused in (False, True):
        x = qkv.clone()
        q, k, v = x.split([H * D] * 3, dim=-1)
        kp, vp = allocate_gpu_cache(N, bs, DEV, dtype=dtype)
        kp.fill_(3)
        vp.fill_(5)
        out = torch.zeros((pad, H * D), dtype=dtype, device=DEV)
        if fused:
            def step():
                torch_ops.rope_prefill_and_cache(out, positions, q, k, v, cos_sin, kp, vp, dslots, 0, cu, lens, D ** -0.5)
            step()
        else:
            ops.rotary_neox(positions, q, k, cos_sin, num_tokens=T)
            ops.reshape_and_cache(k, v, kp, vp, dslots, layer=0, num_tokens=T)
            ops.prefill_causal(out[:T], q[:T], k[:T], v[:T], cu, max(lens), D ** -0.5, H, prompt_lens=lens)
        torch.cuda.synchronize()
        results.append([t.cpu().view(torch.int16) for t in (x, kp, vp, out)])
    for a, b, what in zip(*results, ("qkv rows", "k pool", "v pool", "outputs")):
        assert torch.equal(a, b), f"{what} differ between the one launch and the three kernels"
    launched = _captured_launches(step)
    assert launched == [64 * waves] if waves else len(launched) == 2


@pytest.mark.parametrize("bs,off", [(16, 0), (16, 8), (16, 5), (32, 0), (32, 16), (32, 8), (8, 0)])
def test_prompt_step_pool_writes_of_runs_that_start_anywhere_in_a_block(bs, off):
    """The step operator writes 16 tokens with two stores where they are 16 slots in
    order from a multiple of 16 inside one block: runs that start at, before and
    behind such a multiple, up to the pool's last slot, against the cache write."""
    print(f"[case] prompt step runs bs={bs} off={off}", flush=True)
    from muxserve_amd import torch_ops
    from muxserve_amd.attention import build_cos_sin_cache
    Hq = Hkv = 2
    lens = [160, 48]
    T = sum(lens)
    N = Hkv * ((T + off + bs - 1) // bs)
    slots = torch.empty((T, 1, Hkv), dtype=torch.int64)
    for h in range(Hkv):
        slots[:, 0, h] = h * (N // Hkv) * bs + off + torch.arange(T)
    slots[-16:, 0, 1] = N * bs - 16 + torch.arange(16)                    # the pool's last slots
    qkv = torch.randn((T + (-T) % 8, (Hq + 2 * Hkv) * D), generator=torch.Generator().manual_seed(bs + off)).half().to(DEV)
    positions = torch.arange(T + (-T) % 8, device=DEV)
    cos_sin = build_cos_sin_cache(D, 2048, 10000.0, DEV)
    cu = torch.tensor([0, lens[0], T], dtype=torch.int32, device=DEV)
    results = []
    for fused in (False, True):
        x = qkv.clone()
        q, k, v = x.split([Hq * D, Hkv * D, Hkv * D], dim=-1)
        kp, vp = allocate_gpu_cache(N, bs, DEV, dtype=torch.float16)
        kp.fill_(3)
        vp.fill_(5)
        if fused:
            out = torch.zeros((x.shape[0], Hq * D), dtype=x.dtype, device=DEV)
            torch_ops.rope_prefill_and_cache(out, positions, q, k, v, cos_sin, kp, vp, slots.to(DEV), 0, cu, lens, D ** -0.5)
        else:
            ops.rotary_neox(positions, q, k, cos_sin, num_tokens=T)
            ops.reshape_and_cache(k, v, kp, vp, slots.to(DEV), layer=0, num_tokens=T)
        torch.cuda.synchronize()
        results.append([t.cpu().view(torch.int16) for t in (x, kp, vp)])
    for a, b, what in zip(*results, ("qkv rows", "k pool", "v pool")):
        assert torch.equal(a, b), f"{what} differ from the rotation and the cache write"


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("Hq,Hkv,lens", [(4, 2, [5, 150, 33]), (8, 8, [5, 30, 17] * 12), (20, 20, [128, 33] * 8),
                                         (8, 8, [60, 33] * 40)])
def test_rotary_table_at_any_float_offset(dtype, Hq, Hkv, lens):
    """The cos|sin table is taken at any 4-byte boundary, as the rotary kernel takes
    it, by the small-step cache write and by the prompt step (the last three in one
    launch): rows, pools and outputs bitwise those of an aligned table."""
    print(f"[case] rotary table offset {dtype} {Hq} {Hkv} {len(lens)}", flush=True)
    from muxserve_amd import torch_ops, workloads
    from muxserve_amd.attention import build_cos_sin_cache
    rng = np.random.Generator(np.random.PCG64(3))
    bs, T = 16, sum(lens)
    N = sum((n + bs - 1) // bs for n in lens) * Hkv
    slots, _ = workloads.prefill_slot_mapping(np.array(lens, dtype=np.int32), Hkv, bs, rng.permutation(N))
    dslots, positions = torch.from_numpy(slots).to(DEV), torch.from_numpy(rng.integers(0, 2048, size=T)).to(DEV)
    cu = torch.tensor(np.concatenate([[0], np.cumsum(lens)]), dtype=torch.int32, device=DEV)
    table = build_cos_sin_cache(D, 2048, 10000.0, DEV)
    qkv = torch.randn((T, (Hq + 2 * Hkv) * D), device=DEV).to(dtype)
    results = []
    for offset in (0, 1):
        cos_sin = torch.zeros(table.numel() + 4, device=DEV)[offset:offset + table.numel()].view_as(table).copy_(table)
        got = []
        for step in (False, True):
            x = qkv.clone()
            q, k, v = x.split([Hq * D, Hkv * D, Hkv * D], dim=-1)
            kp, vp = allocate_gpu_cache(N, bs, DEV, dtype=dtype)
            kp.zero_()
            vp.zero_()
            out = torch.zeros((T, Hq * D), dtype=dtype, device=DEV)
            if step:
                torch_ops.rope_prefill_and_cache(out, positions, q, k, v, cos_sin, kp, vp, dslots, 0, cu, lens, D ** -0.5)
            else:
                ops.rope_reshape_and_cache(positions, q, k, v, cos_sin, kp, vp, dslots)
            got += [t.view(torch.int16) for t in (x, kp, vp, out)]
        results.append(got)
    assert all(torch.equal(a, b) for a, b in zip(*results))


@pytest.mark.parametrize("form", ["rotary", "cache write of few", "cache write of many", "short prompts"])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_rotation_rounds_to_nearest_even(dtype, form):
    """Rows that the rotation turns into the table's own floats, so that the stored value is
    one rounding of a chosen float: ties and their neighbours in the last stored bit, the
    largest finite values and past them, subnormals, infinities, NaN, random bits.  x = (1,
    0): x' = cos, y' = sin, bitwise as torch rounds them (any NaN for a NaN)."""
    print(f"[case] rounding {dtype} {form}", flush=True)
    from muxserve_amd import torch_ops
    H, bs = 8, 16
    T = {"rotary": 300, "cache write of few": 300, "cache write of many": 700, "short prompts": 300}[form]
    rng = np.random.Generator(np.random.PCG64(T))
    bits = rng.integers(0, 2 ** 32, size=(T, D // 2), dtype=np.uint64).astype(np.uint32)
    step = 16 if dtype == torch.bfloat16 else 13
    low = np.array([0, 1, (1 << step - 1) - 1, 1 << step - 1, (1 << step - 1) + 1, (1 << step) - 1], dtype=np.uint32)
    bits[1::2] = (bits[1::2] >> step << step) | low[rng.integers(0, len(low), size=bits[1::2].shape)]
    bits[2::6] = (bits[2::6] & 0x807fffff) | (rng.integers(0x67, 0x92, size=bits[2::6].shape).astype(np.uint32) << 23)
    special = np.array([0x7f800000, 0xff800000, 0x7fc00000, 0xffc12345, 0x7f7fffff, 0x7f7f7fff, 0x7f7f8000, 1, 0x80000001,
                        0x00007fff, 0x00008000, 0x00018000, 0x477fefff, 0x477ff000, 0x33000000, 0x33000001], dtype=np.uint32)
    bits[0, :16] = special
    values = torch.from_numpy(bits.view(np.float32))
    zero = torch.zeros_like(values)
    positions = torch.arange(T, device=DEV)
    slots = torch.randperm(T * H, generator=torch.Generator().manual_seed(1)).reshape(T, 1, H).to(DEV)
    one = torch.zeros((T, 3 * H * D), dtype=dtype)
    one.view(T, -1, 2, D // 2)[:, :, 0] = 1
    for half, table in ((0, torch.cat([values, zero], 1)), (1, torch.cat([zero, values], 1))):
        q, k, v = one.to(DEV).split([H * D] * 3, dim=-1)
        cos_sin = table.to(DEV).contiguous()
        kp, vp = allocate_gpu_cache(T * H // bs + 1, bs, DEV, dtype=dtype)
        if form == "rotary":
            ops.rotary_neox(positions, q, k, cos_sin)
        elif form == "short prompts":
            cu = torch.arange(0, T + 1, 30, dtype=torch.int32, device=DEV)
            out = torch.zeros((T, H * D), dtype=dtype, device=DEV)
            torch_ops.rope_prefill_and_cache(out, positions, q, k, v, cos_sin, kp, vp, slots, 0, cu, [30] * 10, 1.0)
        else:
            ops.rope_reshape_and_cache(positions, q, k, v, cos_sin, kp, vp, slots)
        want = values.to(dtype)
        for x in (q, k):
            got = x.cpu().reshape(T, H, 2, D // 2)[:, :, half]
            nan = want.isnan()[:, None].expand_as(got)
            assert torch.equal(got.isnan(), nan)
            same = got.contiguous().view(torch.int16) == want.view(torch.int16)[:, None]
            assert (same | nan).all(), (half, int((~(same | nan)).sum()))


@pytest.mark.parametrize("rope", [True, False])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_multi_model_cache_write_equals_one_launch_per_model(rope, dtype):
    """mux_multi_rope_reshape_and_cache over three colocated models (7B, 13B, a
    grouped-query shape; a decode-shaped step of single tokens for two of them
    and packed ragged prompts for the third, one empty model in between) against
    one call per model: q, k rows and both pools bitwise equal, and the plain
    variant bitwise equal to the oracle's scatter."""
    print(f"[case] multi-model cache write rope={rope} {dtype}", flush=True)
    from oracle import attn_oracle as orc
    from muxserve_amd import workloads
    from muxserve_amd.attention import build_cos_sin_cache
    from muxserve_amd.pool import allocate_gpu_cache
    bs, L, layer = 16, 2, 1
    rng = np.random.Generator(np.random.PCG64(91))
    g = torch.Generator().manual_seed(91)
    shapes = [(32, 32, 32), (40, 40, 16), (8, 2, 0), (16, 4, None)]      # Hq, Hkv, decode tokens (None: prompts)
    lens3 = rng.permutation(np.arange(1, 24)).astype(np.int32)
    need = sum(hk * (t if t is not None else int(((lens3 + bs - 1) // bs).sum())) for _, hk, t in shapes)
    N = need + 11
    ids = rng.permutation(N)
    cos_sin = build_cos_sin_cache(D, 4096, 10000.0, DEV)
    models, cur = [], 0
    for hq, hk, t in shapes:
        if t is None:
            slots1, used = workloads.prefill_slot_mapping(lens3, hk, bs, ids[cur:])
            T = int(lens3.sum())
        else:
            # a decode step: every sequence writes one token somewhere inside its last block
            T = t
            blk = ids[cur:cur + T * hk].reshape(T, hk).astype(np.int64)
            slots1 = (blk * bs + rng.integers(0, bs, size=(T, 1)))[:, None, :]
            used = T * hk
        cur += used
        slots = np.full((T, L, hk), -1, dtype=np.int64)
        slots[:, layer, :] = slots1[:, 0, :]
        if T > 3:
            slots[2, layer, 0] = -1
        pad = (T + 7) // 8 * 8
        qkv = torch.randn((pad, (hq + 2 * hk) * D), generator=g).to(dtype).to(DEV)
        pos = torch.from_numpy(rng.integers(0, 4096, size=pad)).to(DEV)
        models.append((hq, hk, T, qkv, pos, torch.from_numpy(slots).to(DEV), slots))
    results = []
    for fused in (False, True):
        kp, vp = allocate_gpu_cache(N, bs, DEV, dtype=dtype)
        kp.zero_()
        vp.zero_()
        xs, calls = [], []
        for hq, hk, T, qkv, pos, dslots, _ in models:
            x = qkv.clone()
            xs.append(x)
            q, k, v = x.split([hq * D, hk * D, hk * D], dim=-1)
            if fused:
                calls.append(ops.CacheWriteCall(k, v, dslots, layer=layer, positions=pos if rope else None,
                                                cos_sin=cos_sin if rope else None, q=q if rope else None,
                                                num_tokens=T))
            elif rope:
                ops.rope_reshape_and_cache(pos, q, k, v, cos_sin, kp, vp, dslots, layer=layer, num_tokens=T)
            else:
                ops.reshape_and_cache(k, v, kp, vp, dslots, layer=layer, num_tokens=T)
        if fused:
            ops.multi_reshape_and_cache(calls, kp, vp)
        torch.cuda.synchronize()
        results.append(([x.cpu().view(torch.int16) for x in xs], kp.cpu(), vp.cpu()))
    for xa, xb in zip(results[0][0], results[1][0]):
        assert torch.equal(xa, xb), "q/k rows differ between the fused launch and the per-model launches"
    assert torch.equal(results[0][1].view(torch.int16), results[1][1].view(torch.int16))
    assert torch.equal(results[0][2].view(torch.int16), results[1][2].view(torch.int16))
    if not rope:
        hk_pool, hv_pool = orc.allocate_pool(N, bs, dtype)
        hk_pool.zero_()
        hv_pool.zero_()
        for hq, hk, T, qkv, pos, _, slots in models:
            if T == 0:
                continue
            _, k, v = qkv.cpu().split([hq * D, hk * D, hk * D], dim=-1)
            orc.reshape_and_cache(k[:T], v[:T], hk_pool, hv_pool, torch.from_numpy(slots), layer=layer)
        assert torch.equal(results[1][1].view(torch.int16), hk_pool.view(torch.int16))
        assert torch.equal(results[1][2].view(torch.int16), hv_pool.view(torch.int16))


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_decode_layer_operator_equals_the_general_path(dtype):
    """One decode step through PagedAttentionWithRoPE as one operator, with the two
    kernels of large steps (fused_rope_max_tokens 0), and with query rows that
    16-byte accesses cannot take: rows, pools and outputs bitwise equal."""
    print(f"[case] decode layer operator {dtype}", flush=True)
    from muxserve_amd.attention import InputMetadata
    Hq, Hkv, bs, lens = 8, 2, 16, [1, 17, 700, 33, 1100]
    B, nb = len(lens), -(-max(lens) // bs)
    g = torch.Generator().manual_seed(9)
    N = B * Hkv * nb
    tables = torch.randperm(N, generator=g).to(torch.int32).reshape(1, B, Hkv, nb)
    slots = torch.stack([tables[0, i, :, (n - 1) // bs].long() * bs + (n - 1) % bs for i, n in enumerate(lens)])[:, None]
    ctx = torch.tensor(lens, dtype=torch.int32)
    md = InputMetadata(prompt_lens=[], slot_mapping=slots.contiguous().to(DEV), context_lens=ctx.to(DEV),
                       max_context_len=max(lens), block_tables=tables.to(DEV), total_context_len=sum(lens))
    rows = torch.randn((8, (Hq + 2 * Hkv) * D), generator=g).to(dtype)
    kp0 = torch.randn((N, D // 8, bs, 8), generator=g).to(dtype)
    vp0 = torch.randn((N, D, bs), generator=g).to(dtype)
    positions = torch.tensor([n - 1 for n in lens] + [0] * 3, device=DEV)
    results = []
    for fused_max, pad in ((512, 0), (0, 0), (512, 2)):
        layer = PagedAttentionWithRoPE(Hq, D, D ** -0.5, max_position=2048, rotary_dim=D, num_kv_heads=Hkv, layer_idx=0)
        layer.fused_rope_max_tokens = fused_max
        kp, vp = kp0.to(DEV), vp0.to(DEV)
        _, k, v = rows.to(DEV).split([Hq * D, Hkv * D, Hkv * D], dim=-1)
        q = torch.zeros((8, Hq * D + pad), dtype=dtype, device=DEV)[:, pad:]
        q.copy_(rows[:, :Hq * D])
        out = layer(positions, q, k, v, kp, vp, md, None)
        torch.cuda.synchronize()
        results.append([t.cpu().contiguous().view(torch.int16) for t in (out[:B], q, k, kp, vp)])
    for got in results[1:]:
        for a, b, what in zip(results[0], got, ("outputs", "q", "k", "k pool", "v pool")):
            assert torch.equal(a, b), what


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("bs", [8, 16, 32])
@pytest.mark.parametrize("n", [1, 8, 17, 63, 64, 65, 97, 256, 257, 400, 512, 513])
def test_decode_of_one_sequence_in_one_launch_equals_the_general_path(dtype, bs, n):
    """One sequence with as many kv heads as query heads (one launch up to 512 tokens)
    against rotation, cache write and attention in turn: q, k and the pools bitwise, the
    output bitwise while the general path has one workgroup per head (256 tokens) and
    within the rounding of the stored value beyond.  The new token in its place; no slot;
    a slot outside the pool, in an earlier block of the table, in a block that the table
    names twice, and in none of its blocks."""
    print(f"[case] decode of one sequence {dtype} bs={bs} n={n}", flush=True)
    from muxserve_amd.attention import InputMetadata
    H, nb = 8, -(-n // bs)
    g = torch.Generator().manual_seed(n + bs)
    N = H * (nb + 2)
    tables = torch.randperm(N, generator=g).to(torch.int32)
    spare = tables[H * nb:]
    tables = tables[:H * nb].reshape(1, 1, H, nb).clone()
    slots = tables[0, 0, :, nb - 1].long() * bs + (n - 1) % bs
    slots[1] = -1
    slots[2] = N * bs
    slots[3] = tables[0, 0, 3, 0].long() * bs + min(bs - 1, n - 1) // 2
    tables[0, 0, 4, nb // 2] = tables[0, 0, 4, nb - 1]
    slots[5] = spare[0].long() * bs + bs - 1
    ctx = torch.tensor([n], dtype=torch.int32)
    md = InputMetadata(prompt_lens=[], slot_mapping=slots[None, None].contiguous().to(DEV), context_lens=ctx.to(DEV),
                       max_context_len=n, block_tables=tables.to(DEV), total_context_len=n, context_lens_host=ctx)
    rows = torch.randn((8, 3 * H * D), generator=g).to(dtype)
    kp0 = torch.randn((N, D // 8, bs, 8), generator=g).to(dtype)
    vp0 = torch.randn((N, D, bs), generator=g).to(dtype)
    positions = torch.tensor([n - 1] + [0] * 7, device=DEV)
    results = []
    for fused_max in (512, 0):
        layer = PagedAttentionWithRoPE(H, D, D ** -0.5, max_position=2048, rotary_dim=D, num_kv_heads=H, layer_idx=0)
        layer.fused_rope_max_tokens = fused_max
        kp, vp, x = kp0.to(DEV), vp0.to(DEV), rows.to(DEV)
        q, k, v = x.split([H * D] * 3, dim=-1)
        out = layer(positions, q, k, v, kp, vp, md, None)
        torch.cuda.synchronize()
        results.append([t.cpu() for t in (x, kp, vp, out[:1])])
        if fused_max:
            launched = _captured_launches(lambda: layer(positions, q, k, v, kp, vp, md, None))
            assert launched == [256 if n <= 256 else 512] if n <= 512 else len(launched) > 1
    for a, b, what in zip(*results, ("q, k, v", "k pool", "v pool")):
        assert torch.equal(a.view(torch.int16), b.view(torch.int16)), what
    got, want = (r[3].float() for r in results)
    # Beyond 256 tokens the waves hold other tokens, so their maxima differ, and f16
    # probabilities, relative to them, round differently: 2^-11 of each weight on either
    # side, at most 2^-10 max |v| in their mean.  bf16 keeps them in 32 bits (sums in
    # another order).  Then the rounding of the stored value.
    if n <= 256:
        bound = torch.zeros_like(want)
    elif dtype == torch.float16:
        bound = want.abs() * 2.0 ** -10 + 2.0 ** -10 * float(vp0.abs().max())
    else:
        bound = want.abs() * 2.0 ** -7 + 1e-5
    assert ((got - want).abs() <= bound).all(), (got - want).abs().max()


@pytest.mark.parametrize("n", [40, 600])
def test_prompt_step_with_unaligned_query_rows_is_refused(n):
    """The attention kernel takes 16-byte accesses to the query rows only; such a
    step reaches the general path, which refuses it, whatever its size."""
    from muxserve_amd.attention import InputMetadata
    H, bs = 2, 16
    nb = -(-n // bs)
    kp, vp = allocate_gpu_cache(nb * H, bs, DEV)
    t = torch.arange(n, device=DEV)
    slots = torch.stack([(t // bs * H + h) * bs + t % bs for h in range(H)], dim=1)[:, None].contiguous()
    none = torch.empty((0,), dtype=torch.int32, device=DEV)
    md = InputMetadata(prompt_lens=[n], slot_mapping=slots, context_lens=none, max_context_len=0,
                       block_tables=none.view(0, 0, 0, 0))
    layer = PagedAttentionWithRoPE(H, D, D ** -0.5, max_position=2048, rotary_dim=D, num_kv_heads=H, layer_idx=0)
    k, v = (torch.randn((n, H * D), device=DEV).half() for _ in range(2))
    q = torch.zeros((n, H * D + 2), dtype=torch.float16, device=DEV)[:, 2:]
    with pytest.raises(RuntimeError, match="invalid argument"):
        layer(t, q, k, v, kp, vp, md, None)


def test_empty_steps_are_accepted():
    """No tokens, no sequences, no prompts, no sampled rows: every entry point
    returns without launching and without touching its outputs."""
    print("[case] empty steps", flush=True)
    from muxserve_amd.attention import build_cos_sin_cache
    H, bs, N = 2, 16, 64
    k_pool, v_pool = allocate_gpu_cache(N, bs, DEV)
    k_pool.fill_(3.0)
    v_pool.fill_(3.0)
    e16 = torch.empty((0, H * D), dtype=torch.float16, device=DEV)
    slots = torch.empty((0, 1, H), dtype=torch.int64, device=DEV)
    pos = torch.empty((0,), dtype=torch.int64, device=DEV)
    cos_sin = build_cos_sin_cache(D, 64, 10000.0, DEV)
    ops.reshape_and_cache(e16, e16, k_pool, v_pool, slots)
    ops.rotary_neox(pos, e16, e16, cos_sin)
    ops.rope_reshape_and_cache(pos, e16, e16, e16, cos_sin, k_pool, v_pool, slots)
    # a padded batch whose valid part is empty
    pad = torch.full((8, H * D), 5.0, dtype=torch.float16, device=DEV)
    ops.reshape_and_cache(pad, pad, k_pool, v_pool, torch.zeros((8, 1, H), dtype=torch.int64, device=DEV), num_tokens=0)
    out = torch.full((8, H * D), 7.0, dtype=torch.float16, device=DEV)
    ops.paged_decode(out, pad, k_pool, v_pool, torch.empty((1, 0, H, 4), dtype=torch.int32, device=DEV),
                     torch.empty((0,), dtype=torch.int32, device=DEV), 0, D ** -0.5)
    ops.prefill_causal(out, pad, pad, pad, torch.zeros((1,), dtype=torch.int32, device=DEV), 0, D ** -0.5, H)
    assert ops.rms_norm(e16[:, :64], torch.ones((64,), dtype=torch.float16, device=DEV), 1e-6).shape == (0, 64)
    assert ops.silu_and_mul(e16).shape == (0, H * D // 2)
    emb = torch.zeros((32, 256), dtype=torch.float16, device=DEV)
    assert ops.greedy_sample(emb, torch.zeros((8, 256), dtype=torch.float16, device=DEV), 32, 0).shape == (0,)
    torch.cuda.synchronize()
    assert (out == 7.0).all() and (k_pool == 3.0).all() and (v_pool == 3.0).all()
