"""What the speed of this package is measured on: one pass through its public
entry points per case, over the sizes a serving loop gives them.

  decode    the attention of one decode step, one layer: rotary embedding of q
            and k, KV-cache write of the new tokens, paged attention.  One model:
            PagedAttentionWithRoPE.forward.  Several colocated models: the two
            fused launches (multi_reshape_and_cache, DecodeLaunch).
  prefill   the same for a step of prompts (causal attention).
  sample    GreedySampler.forward: lm_head product, argmax, tokens on the host.
  norm_act  the RMSNorm of the residual stream and the SiluAndMul of the MLP.
  steps     prepare_inputs: a batch of requests arrives, is prefilled, decodes
            16 tokens and leaves; what is timed is the building of the index
            tensors of those 17 steps.

Block ids are a random draw from a pool of at least half a million blocks (what
a pool that several models have shared for a while hands out); the index
tensors hold four layers, of which a pass uses one.
"""
import math
import random

import numpy as np
import torch

from muxserve_amd import ops, workloads
from muxserve_amd.attention import InputMetadata, PagedAttentionWithRoPE, build_cos_sin_cache
from muxserve_amd.batch_scheduler import BatchScheduler
from muxserve_amd.device_tables import DeviceBlockTables
from muxserve_amd.layers import GreedySampler, RMSNorm, SiluAndMul
from muxserve_amd.memory_manager import KVStorage
from muxserve_amd.pool import HEAD_SIZE, allocate_gpu_cache
from muxserve_amd.prepare import prepare_inputs

DEV = "cuda:0"
D = HEAD_SIZE
LAYERS, LAYER = 4, 2                 # layers of the index tensors, and the one in use
MIN_POOL_BLOCKS = 1 << 19
MAX_POSITION = 8192
VOCAB = 32000
DECODE_STEPS = 16
DTYPES = {"f16": torch.float16, "bf16": torch.bfloat16}
# hidden size (query heads x head size) follows from workloads.LLAMA_SHAPES; the
# width of the MLP:
MLP_WIDTH = {"7b": 11008, "13b": 13824, "30b": 17920, "65b": 22016, "70b-gqa": 28672}


def listed():
    return [
        # One user, one model: a chat reply streams out a token at a time.
        _attn("decode_7b_single", "decode", "7b", "1", median=97, lo=97, hi=97),
        # An ordinary batch of one model in bf16.
        _attn("decode_13b_b16_bf16", "decode", "13b", "16", dtype="bf16", median=300, sigma=0.8, lo=16, hi=2048),
        # Three colocated models of different head counts: the mix this package is built for.
        _attn("decode_mixed3", "decode", "7b+13b+30b", "32+16+8", median=300, sigma=0.8, lo=16, hi=2048),
        # A popular model at a large batch.
        _attn("decode_7b_b256", "decode", "7b", "256", median=300, sigma=0.8, lo=16, hi=2048),
        # Long documents on a grouped-query model: the most K/V a step reads here.
        _attn("decode_70b_gqa_long_bf16", "decode", "70b-gqa", "64", dtype="bf16", lo=2048, hi=8192),
        # One short question arrives.
        _attn("prefill_7b_single", "prefill", "7b", "1", median=45, lo=45, hi=45),
        # The prompts of three colocated models, ragged as users write them.
        _attn("prefill_mixed3", "prefill", "7b+13b+30b", "16+16+16", median=200, sigma=1.0, lo=8, hi=2048),
        # Full-length prompts.
        _attn("prefill_7b_long", "prefill", "7b", "16", median=2048, lo=2048, hi=2048),
        # A few long prompts of odd lengths on a grouped-query model in bf16.
        _attn("prefill_70b_gqa_bf16", "prefill", "70b-gqa", "3", dtype="bf16", lo=700, hi=4000),
        # The tokens of the large decode batch.
        {"name": "sample_7b_b256", "kind": "sample", "models": "7b", "dtype": "f16", "rows": 256, "prompt_step": False},
        # The element-wise operators of a prefill step.
        {"name": "norm_act_30b_prefill", "kind": "norm_act", "models": "30b", "dtype": "f16", "rows": 4096},
        # The index tensors of a batch of requests over its life.
        {"name": "steps_7b_b32", "kind": "steps", "models": "7b", "batch": "32", "block": 16, "median": 300,
         "sigma": 0.8, "lo": 16, "hi": 1024, "lens_seed": 5},
    ]


def _attn(name, kind, models, batch, dtype="f16", block=16, median=0, sigma=0.0, lo=1, hi=1, lens_seed=3):
    """median 0: lengths uniform in [lo, hi]; else lognormal, clipped to them."""
    return {"name": name, "kind": kind, "models": models, "batch": batch, "dtype": dtype, "block": block,
            "median": median, "sigma": sigma, "lo": lo, "hi": hi, "lens_seed": lens_seed}


def _log_int(rng, lo, hi):
    return min(hi, max(lo, round(math.exp(rng.uniform(math.log(lo), math.log(hi))))))


def draw(rng):
    kind = rng.choice(["decode"] * 4 + ["prefill"] * 4 + ["sample", "sample", "norm_act", "steps"])
    dtype = rng.choice(["f16", "bf16"])
    model = rng.choice(["7b", "13b", "30b", "65b", "70b-gqa", "70b-gqa"])
    if kind == "sample":
        return {"kind": kind, "models": model, "dtype": dtype, "rows": _log_int(rng, 1, 256),
                "prompt_step": rng.random() < 0.3}
    if kind == "norm_act":
        return {"kind": kind, "models": model, "dtype": dtype, "rows": _log_int(rng, 1, 2048)}
    if kind == "steps":
        return {"kind": kind, "models": rng.choice(["7b", "13b"]), "batch": str(_log_int(rng, 1, 32)), "block": 16,
                "median": _log_int(rng, 50, 300), "sigma": 0.8, "lo": 16, "hi": 1024,
                "lens_seed": rng.randrange(1 << 20)}
    if rng.random() < 0.3:
        model = rng.choice(["7b+13b", "13b+30b", "7b+13b+30b", "7b+7b"])
    n = len(model.split("+"))
    block = rng.choice([16, 16, 16, 16, 8, 32])
    seed = rng.randrange(1 << 20)
    longest = 8192 if kind == "decode" else 4096
    median, sigma = _log_int(rng, 30, longest // 2), rng.choice([0.0, 0.5, 0.8, 1.0])
    batch = [_log_int(rng, 1, 256 if kind == "decode" else 24) for _ in range(n)]
    while True:
        c = _attn("", kind, model, "+".join(map(str, batch)), dtype, block, median, sigma, 1, longest, seed)
        del c["name"]
        w = work(c)
        if w["bytes"] <= 1.2e9 and w["flops"] <= (1e18 if kind == "decode" else 2.5e11):
            return c
        if max(batch) == 1:
            median = c["median"] = median // 2
        batch = [max(1, b // 2) for b in batch]


# ---- sizes ---------------------------------------------------------------------------

def _shapes(case):
    return [workloads.LLAMA_SHAPES[m] for m in case["models"].split("+")]


def _lengths(case):
    """Context or prompt lengths per model: part of the case, not of the seed."""
    rng = random.Random(case["lens_seed"])
    out = []
    for b in case["batch"].split("+"):
        if case["median"]:
            lens = [round(rng.lognormvariate(math.log(case["median"]), case["sigma"])) for _ in range(int(b))]
        else:
            lens = [rng.randint(case["lo"], case["hi"]) for _ in range(int(b))]
        out.append([min(case["hi"], max(case["lo"], n)) for n in lens])
    return out


def work(case):
    kind = case["kind"]
    if kind in ("decode", "prefill"):
        nbytes = flops = 0
        for (hq, hkv, _), lens in zip(_shapes(case), _lengths(case)):
            tokens = len(lens) if kind == "decode" else sum(lens)
            # q, k, v read; q, k rotated in place; k, v to the pool, a slot per (token, head); the output
            nbytes += tokens * (D * 2 * ((hq + 2 * hkv) + (hq + hkv) + 2 * hkv + hq) + 8 * hkv + 8 + 4 * D)
            if kind == "decode":
                nbytes += sum(2 * n * hkv * D * 2 + 4 * hkv * -(-n // case["block"]) + 4 for n in lens)
                flops += 4 * hq * D * sum(lens)
            else:
                flops += 4 * hq * D * sum(n * (n + 1) // 2 for n in lens)
        return {"bytes": nbytes, "flops": flops}
    hq = _shapes(case)[0][0]
    if kind == "sample":
        return {"bytes": VOCAB * hq * D * 2 + case["rows"] * (hq * D * 2 + 8), "flops": 2 * VOCAB * hq * D * case["rows"]}
    if kind == "norm_act":
        width = MLP_WIDTH[case["models"]]
        return {"bytes": case["rows"] * (2 * hq * D + 3 * width) * 2, "flops": 0}
    _, heads, layers = _shapes(case)[0]
    lens = _lengths(case)[0]
    nbytes = sum(lens) * layers * heads * 8
    for s in range(1, DECODE_STEPS + 1):
        blocks = max(-(-(n + s) // case["block"]) for n in lens)
        nbytes += len(lens) * layers * heads * (8 + 4 * blocks)
    return {"bytes": nbytes, "flops": 0}


def tolerance(case):
    kind = case["kind"]
    if kind == "steps":
        return "exact"                       # integers
    if kind == "sample":
        return {"rel": 0.0, "differ": 0.005}  # tokens: ties of the rounded logits
    # About four times what the attention outputs and the rotated q and k differ
    # from the same arithmetic in 64 bits (f16: rel 2.8e-4, max 3.7e-3; bf16:
    # 1.7e-3 and 3.9e-3, the rounding of the stored values).
    if case["dtype"] == "f16":
        return {"rel": 1.1e-3, "max": 0.015}
    return {"rel": 6.5e-3, "max": 0.016}


# ---- states --------------------------------------------------------------------------

_kept = {}                                   # what a program makes once and keeps: its layers


def _layer(hq, hkv):
    key = (hq, hkv)
    if key not in _kept:
        _kept[key] = PagedAttentionWithRoPE(hq, D, D ** -0.5, base=10000, max_position=MAX_POSITION, rotary_dim=D,
                                            num_kv_heads=hkv, rope_scaling=None, layer_idx=LAYER)
    return _kept[key]


def _cos_sin():
    if "cos_sin" not in _kept:
        _kept["cos_sin"] = build_cos_sin_cache(D, MAX_POSITION, 10000.0, DEV)
    return _kept["cos_sin"]


def prepare(case, seed):
    g = torch.Generator(device=DEV).manual_seed(seed)
    return {"decode": _prepare_attention, "prefill": _prepare_attention, "sample": _prepare_sample,
            "norm_act": _prepare_norm_act, "steps": _prepare_steps}[case["kind"]](case, g, seed)


def _normal(shape, dtype, g, scale=1.0):
    return torch.empty(shape, dtype=dtype, device=DEV).normal_(0.0, scale, generator=g)


def _prepare_attention(case, g, seed):
    bs, dtype, decode = case["block"], DTYPES[case["dtype"]], case["kind"] == "decode"
    lengths, shapes = _lengths(case), _shapes(case)
    need = sum(hkv * sum(-(-n // bs) for n in lens) for (_, hkv, _), lens in zip(shapes, lengths))
    pool_blocks = max(MIN_POOL_BLOCKS * 16 // bs, 2 * need)
    k_pool, v_pool = allocate_gpu_cache(pool_blocks, bs, DEV, dtype)
    k_pool.normal_(generator=g)
    v_pool.normal_(generator=g)
    ids = torch.randperm(pool_blocks, generator=g, device=DEV)[:need]
    models, at = [], 0
    for (hq, hkv, _), lens in zip(shapes, lengths):
        n = torch.tensor(lens, device=DEV)
        blocks = (n + bs - 1) // bs
        width = -(-max(lens) // bs)
        used = (torch.arange(width, device=DEV) < blocks[:, None, None]).expand(len(lens), hkv, width)
        table = torch.full((len(lens), hkv, width), -1, dtype=torch.int64, device=DEV)
        count = hkv * sum(-(-x // bs) for x in lens)
        table[used] = ids[at:at + count]
        at += count
        if decode:                           # the newest token of every sequence
            row, positions = torch.arange(len(lens), device=DEV), n - 1
        else:                                # every token of every prompt
            row = torch.repeat_interleave(torch.arange(len(lens), device=DEV), n)
            starts = torch.cumsum(n, 0) - n
            positions = torch.arange(sum(lens), device=DEV) - starts[row]
        slots = table[row, :, positions // bs] * bs + (positions % bs)[:, None]
        tokens = positions.numel()
        padded = (tokens + 7) // 8 * 8
        pos = torch.zeros((padded,), dtype=torch.int64, device=DEV)
        pos[:tokens] = positions
        qkv = _normal((padded, (hq + 2 * hkv) * D), dtype, g)
        q, k, v = qkv.split([hq * D, hkv * D, hkv * D], dim=-1)
        m = {"hq": hq, "hkv": hkv, "lens": lens, "tokens": tokens, "positions": pos, "qkv": qkv, "q": q, "k": k, "v": v,
             "slots": slots[:, None, :].repeat(1, LAYERS, 1).contiguous()}
        if decode:
            m["tables"] = table.to(torch.int32)[None].repeat(LAYERS, 1, 1, 1).contiguous()
            m["context_lens"] = n.to(torch.int32)
            m["context_lens_host"] = torch.tensor(lens, dtype=torch.int32)
        models.append(m)
    s = {"kind": case["kind"], "k_pool": k_pool, "v_pool": v_pool, "models": models}
    if len(models) == 1:
        m = models[0]
        s["layer"] = _layer(m["hq"], m["hkv"])
        if decode:
            s["metadata"] = InputMetadata(prompt_lens=[], slot_mapping=m["slots"], context_lens=m["context_lens"],
                                          max_context_len=max(m["lens"]), block_tables=m["tables"],
                                          total_context_len=sum(m["lens"]), context_lens_host=m["context_lens_host"])
        else:
            s["metadata"] = InputMetadata(prompt_lens=m["lens"], slot_mapping=m["slots"],
                                          context_lens=torch.empty((0,), dtype=torch.int32, device=DEV),
                                          max_context_len=0,
                                          block_tables=torch.empty((0, 0, 0, 0), dtype=torch.int32, device=DEV))
        return s
    # Several models: the descriptors of a step, which a serving loop makes once per step.
    for m in models:
        m["out"] = torch.zeros((m["qkv"].shape[0], m["hq"] * D), dtype=dtype, device=DEV)
    s["writes"] = [ops.CacheWriteCall(m["k"], m["v"], m["slots"], LAYER, m["positions"], _cos_sin(), m["q"], m["tokens"])
                   for m in models]
    if decode:
        s["attention"] = ops.DecodeLaunch(
            [ops.DecodeCall(m["out"], m["q"], m["tables"], m["context_lens"], max(m["lens"]), D ** -0.5, LAYER,
                            sum(m["lens"]), m["context_lens_host"]) for m in models], k_pool, v_pool)
    else:
        calls = []
        for m in models:
            cu = torch.tensor(np.concatenate([[0], np.cumsum(m["lens"])]), dtype=torch.int32, device=DEV)
            calls.append(ops.PrefillCall(m["out"], m["q"], m["k"], m["v"], cu, m["lens"], D ** -0.5, m["hkv"]))
        s["attention"] = calls
    return s


def _prepare_sample(case, g, seed):
    hidden, dtype, rows = _shapes(case)[0][0] * D, DTYPES[case["dtype"]], case["rows"]
    none = torch.empty((0, 0, 0), dtype=torch.int64, device=DEV)
    if case["prompt_step"]:                  # the last row of every prompt
        lens = [random.Random(i).randint(5, 40) for i in range(rows)]
        context_lens = torch.empty((0,), dtype=torch.int32, device=DEV)
    else:
        lens, context_lens = [], torch.ones((rows,), dtype=torch.int32, device=DEV)
    tokens = sum(lens) if lens else rows
    md = InputMetadata(prompt_lens=lens, slot_mapping=none, context_lens=context_lens, max_context_len=0,
                       block_tables=torch.empty((0, 0, 0, 0), dtype=torch.int32, device=DEV))
    return {"kind": "sample", "sampler": GreedySampler(VOCAB), "metadata": md,
            "lm_head": _normal((VOCAB, hidden), dtype, g, 0.05),
            "hidden": _normal(((tokens + 7) // 8 * 8, hidden), dtype, g)}


def _prepare_norm_act(case, g, seed):
    hidden, dtype, rows = _shapes(case)[0][0] * D, DTYPES[case["dtype"]], case["rows"]
    norm = RMSNorm(hidden, eps=1e-6).to(device=DEV, dtype=dtype)
    with torch.no_grad():
        norm.weight.copy_(1 + _normal((hidden,), dtype, g, 0.1))
    return {"kind": "norm_act", "norm": norm, "act": SiluAndMul(), "x": _normal((rows, hidden), dtype, g),
            "gate_up": _normal((rows, 2 * MLP_WIDTH[case["models"]]), dtype, g)}


def _prepare_steps(case, g, seed):
    _, heads, layers = _shapes(case)[0]
    lens, bs = _lengths(case)[0], case["block"]
    longest = 2048
    scheduler = BatchScheduler(layers, heads, longest, bs)
    storage = KVStorage(sum((n + DECODE_STEPS) // bs + 2 for n in lens) * layers * heads)
    rng = np.random.Generator(np.random.PCG64(seed))
    return {"kind": "steps", "scheduler": scheduler, "storage": storage, "layers": layers, "heads": heads,
            "tables": DeviceBlockTables(scheduler, len(lens), DEV),
            "prompts": [rng.integers(0, VOCAB, size=n).astype(np.int32) for n in lens],
            "tokens": [[int(t) for t in rng.integers(0, VOCAB, size=len(lens))] for _ in range(DECODE_STEPS)]}


# ---- one pass --------------------------------------------------------------------------

def run(s):
    kind = s["kind"]
    if kind == "sample":
        return np.asarray(s["sampler"](s["lm_head"], s["hidden"], s["metadata"]))
    if kind == "norm_act":
        return {"norm": s["norm"](s["x"]), "act": s["act"](s["gate_up"])}
    if kind == "steps":
        return _run_steps(s)
    models, k_pool, v_pool = s["models"], s["k_pool"], s["v_pool"]
    if len(models) == 1:
        m = models[0]
        out = s["layer"](m["positions"], m["q"], m["k"], m["v"], k_pool, v_pool, s["metadata"], None)
        outs = [out[:m["tokens"]]]
    else:
        ops.multi_reshape_and_cache(s["writes"], k_pool, v_pool)
        if kind == "decode":
            s["attention"].launch()
        else:
            ops.multi_prefill_causal(s["attention"])
        outs = [m["out"] for m in models]
    return {"out": outs, "qkv": [m["qkv"] for m in models], "k_pool": k_pool, "v_pool": v_pool}


def _run_steps(s):
    scheduler, storage = s["scheduler"], s["storage"]
    ids = list(range(len(s["prompts"])))

    def allocate(request):
        return storage.allocate_batch(request, s["layers"], s["heads"])

    for i in ids:
        scheduler.add_request(s["prompts"][i], i, DECODE_STEPS + 1)
    tokens, positions, md, _, _ = prepare_inputs(scheduler, allocate, ids, [], DEV, device_tables=s["tables"])
    out = {"prefill": [tokens[:md.num_valid_tokens], positions[:md.num_valid_tokens], md.slot_mapping]}
    for last in s["tokens"]:
        tokens, positions, md, _, _ = prepare_inputs(scheduler, allocate, ids, last, DEV, device_tables=s["tables"])
    out["decode"] = [tokens[:len(ids)], positions[:len(ids)], md.slot_mapping, md.block_tables, md.context_lens]
    scheduler.release_requests(ids)
    storage.free_batch(ids)
    return out
