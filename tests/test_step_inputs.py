"""The compact step (get_batch_compact + the device-side builder) against the
reference-shaped step (get_batch), on the host: descriptors are replayed with a
numpy restatement of the three device kernels and must reproduce the oracle's
slot_mapping and block table exactly, through prefill, decode across block
boundaries, release and row reuse, and allocator preemption."""
import numpy as np
import pytest
import torch

from oracle import host_oracle
from muxserve_amd.batch_scheduler import BatchScheduler
from muxserve_amd.memory_manager import KVStorage

D = BatchScheduler.STEP_DESC_INTS


class NumpyMirror:
    """What mux_build_step_inputs does, in numpy."""

    def __init__(self, rows, max_blocks, L, H, bs):
        self.m = np.zeros((rows, max_blocks, L * H), dtype=np.int32)
        self.L, self.H, self.bs = L, H, bs

    def build(self, desc, block_info, num_tokens, max_blocks_out):
        per = self.L * self.H
        for d in desc:
            row, nblk, first, new, off = (int(x) for x in d[:5])
            self.m[row, first:first + new] = block_info[off:off + new * per].reshape(new, per)
        slots = np.zeros((num_tokens, per), dtype=np.int64)
        for d in desc:
            row, nblk, _, _, _, length, t0, dec = (int(x) for x in d)
            if dec:
                slots[t0] = self.m[row, nblk - 1].astype(np.int64) * self.bs + (length - 1) % self.bs
            else:
                for k in range(length):
                    slots[t0 + k] = self.m[row, k // self.bs].astype(np.int64) * self.bs + k % self.bs
        tables = None
        if max_blocks_out > 0:
            tables = np.zeros((self.L, len(desc), self.H, max_blocks_out), dtype=np.int32)
            for c, d in enumerate(desc):
                nblk = int(d[1])
                tables[:, c, :, :nblk] = self.m[int(d[0]), :nblk].reshape(nblk, self.L, self.H).transpose(1, 2, 0)
        return slots.reshape(num_tokens, self.L, self.H), tables


def _compact_step(sched, storage, mirror, L, H, ids, last):
    info = sched.try_batch(list(ids), list(last))
    req = np.ascontiguousarray(info[:-1])
    block_info = (np.asarray(storage.allocate_batch(req, L, H), dtype=np.int32) if int(info[-1]) > 0
                  else np.array([len(ids)], dtype=np.int32))
    bi = sched.get_batch_info(req, block_info)
    T, C, max_ctx, max_blk = bi[:4]
    pad = (T + 7) // 8 * 8
    tok, pos = torch.full((pad,), -7, dtype=torch.int32), torch.full((pad,), -7, dtype=torch.int32)
    ctx = torch.full((C,), -7, dtype=torch.int32)
    n = max(int(block_info[0]), 0)
    desc = torch.full((n, D), -7, dtype=torch.int32)
    sched.get_batch_compact(req, block_info, tok, pos, ctx, desc)
    slots, tables = mirror.build(desc.numpy(), block_info, T, max_blk if max_ctx > 0 else 0)
    return {"tok": tok.long(), "pos": pos.long(), "ctx": ctx, "slots": slots, "tables": tables, "desc": desc.numpy(),
            "batch_reqs": sched.get_batch_reqs(), "preempted": sched.get_preempt_requests(),
            "prompt_info": sched.get_prompt_info()}


def _same(ref, got, bs):
    assert torch.equal(ref["input_tensor"], got["tok"]) and torch.equal(ref["input_positions"], got["pos"])
    assert torch.equal(ref["context_lens"], got["ctx"])
    assert np.array_equal(ref["slot_mapping"].numpy(), got["slots"])
    assert ref["batch_reqs"] == got["batch_reqs"] and ref["preempted_reqs"] == got["preempted"]
    if ref["max_context_len"] > 0:
        rt = ref["block_tables"].numpy()
        for c, n_ctx in enumerate(ref["context_lens"].tolist()):
            valid = (n_ctx + bs - 1) // bs
            assert np.array_equal(rt[:, c, :, :valid], got["tables"][:, c, :, :valid])
            assert (got["tables"][:, c, :, valid:] == 0).all()
    else:
        assert got["tables"] is None


@pytest.mark.parametrize("L,H,bs", [(2, 3, 16), (1, 1, 8), (4, 2, 32)])
def test_compact_step_reproduces_the_reference_step(L, H, bs):
    rng = np.random.Generator(np.random.PCG64(L * 100 + H))
    N = 4000
    ref_store, ref_sched = host_oracle.KVStorage(N), host_oracle.BatchScheduler(L, H, 512, bs)
    store, sched = KVStorage(N), BatchScheduler(L, H, 512, bs)
    sched.enable_device_rows(6)
    mirror = NumpyMirror(6, sched.max_blocks_per_seq, L, H, bs)
    lens = [5, bs, bs + 1, 3 * bs - 1, 1]
    for i, p in enumerate(lens):
        prompt = rng.integers(0, 1000, size=p).astype(np.int32)
        ref_sched.add_request(prompt, i, 64)
        sched.add_request(prompt, i, 64)
    ids = list(range(len(lens)))
    _same(host_oracle.prepare_inputs(ref_sched, ref_store, L, H, ids, []),
          _compact_step(sched, store, mirror, L, H, ids, []), bs)
    order = [3, 0, 4, 1, 2]
    for step in range(2 * bs + 3):                       # every sequence crosses block boundaries
        last = [100 + step] * 5
        got = _compact_step(sched, store, mirror, L, H, order, last)
        _same(host_oracle.prepare_inputs(ref_sched, ref_store, L, H, order, last), got, bs)
        assert sorted(int(d[0]) for d in got["desc"]) == [0, 1, 2, 3, 4]        # rows are stable
    # two requests finish; their rows are reused by new requests
    for s_, st_ in ((ref_sched, ref_store), (sched, store)):
        st_.free_batch([1, 3])
        s_.release_requests([1, 3])
    for rid, p in ((10, 2 * bs), (11, 7), (12, 9)):
        prompt = rng.integers(0, 1000, size=p).astype(np.int32)
        ref_sched.add_request(prompt, rid, 64)
        sched.add_request(prompt, rid, 64)
    got = _compact_step(sched, store, mirror, L, H, [10, 11, 12], [])
    _same(host_oracle.prepare_inputs(ref_sched, ref_store, L, H, [10, 11, 12], []), got, bs)
    assert sorted(int(d[0]) for d in got["desc"]) == [1, 3, 5]
    for step in range(bs + 2):
        idsd = [0, 10, 2, 11, 4, 12]
        last = [7] * 6
        _same(host_oracle.prepare_inputs(ref_sched, ref_store, L, H, idsd, last),
              _compact_step(sched, store, mirror, L, H, idsd, last), bs)
    with pytest.raises(MemoryError):                     # a seventh live request finds no row
        sched.add_request(np.arange(3, dtype=np.int32), 99, 8)
        _compact_step(sched, store, mirror, L, H, [99], [])


def test_compact_step_with_allocator_preemption():
    """A pool too small for the batch: the allocator cuts the batch, the cut
    requests are forgotten and their rows come back."""
    L, H, bs = 2, 2, 16
    per = L * H
    N = 9 * per                                          # room for 9 token blocks in all
    ref_store, ref_sched = host_oracle.KVStorage(N), host_oracle.BatchScheduler(L, H, 256, bs)
    store, sched = KVStorage(N), BatchScheduler(L, H, 256, bs)
    sched.enable_device_rows(4)
    mirror = NumpyMirror(4, sched.max_blocks_per_seq, L, H, bs)
    for i, p in enumerate([3 * bs, 3 * bs, 2 * bs + 5, 2 * bs]):
        prompt = np.arange(p, dtype=np.int32)
        ref_sched.add_request(prompt, i, 32)
        sched.add_request(prompt, i, 32)
    ref = host_oracle.prepare_inputs(ref_sched, ref_store, L, H, [0, 1, 2, 3], [])
    got = _compact_step(sched, store, mirror, L, H, [0, 1, 2, 3], [])
    assert ref["preempted_reqs"] and ref["preempted_reqs"] == got["preempted"]
    _same(ref, got, bs)
    alive = [r for r in [0, 1, 2, 3] if r not in ref["preempted_reqs"]]
    for step in range(bs + 1):                           # decode until the pool runs dry again
        last = [5] * len(alive)
        ref = host_oracle.prepare_inputs(ref_sched, ref_store, L, H, alive, last)
        got = _compact_step(sched, store, mirror, L, H, alive, last)
        _same(ref, got, bs)
        alive = [r for r in alive if r not in ref["preempted_reqs"]]
        if not alive:
            break
    assert sched.num_requests() == ref_sched.num_requests() if hasattr(ref_sched, "num_requests") else True


def test_compact_step_needs_rows_enabled():
    sched = BatchScheduler(1, 1, 64, 16)
    sched.add_request(np.arange(4, dtype=np.int32), 0, 4)
    store = KVStorage(64)
    info = sched.try_batch([0], [])
    req = np.ascontiguousarray(info[:-1])
    blk = store.allocate_batch(req, 1, 1)
    sched.get_batch_info(req, blk)
    with pytest.raises(ValueError):
        sched.get_batch_compact(req, blk, torch.zeros(8, dtype=torch.int32), torch.zeros(8, dtype=torch.int32),
                                torch.zeros(0, dtype=torch.int32), torch.zeros((1, D), dtype=torch.int32))


@pytest.mark.parametrize("blocks,cap", [(40, 0), (40, 3), (9, 0), (9, 1 << 12)])
def test_step_in_one_call_equals_its_four(blocks, cap):
    """BatchScheduler.step against get_batch_info, get_batch_compact,
    get_preempt_requests and get_batch_reqs on a second scheduler: prompts, decode steps
    across block boundaries, preemption (9 token blocks), a staging buffer that has to
    grow (which must not move the step on) and what an unknown request raises."""
    L, H, bs = 2, 3, 16
    pair = []
    for _ in range(2):
        store, sched = KVStorage(blocks * L * H), BatchScheduler(L, H, 256, bs)
        sched.enable_device_rows(4)
        for i, p in enumerate([3 * bs, 2 * bs + 1, bs, 3]):
            sched.add_request(np.arange(p, dtype=np.int32) + i, i, 20 + i)
        pair.append((store, sched))
    buffers = [torch.full((cap,), -5, dtype=torch.int32)]

    def staging(n):
        if buffers[-1].numel() < n:
            buffers.append(torch.full((n,), -5, dtype=torch.int32))
        return buffers[-1]

    alive, last = [0, 1, 2, 3], []
    for step in range(2 * bs + 2):
        got = []
        for store, sched in pair:
            info = sched.try_batch(alive, last)
            req = np.ascontiguousarray(info[:-1])
            reply = store.allocate_batch(req, L, H) if int(info[-1]) > 0 else np.array([len(alive)], dtype=np.int32)
            got.append((sched, req, reply))
        (sched, req, reply), (one, req1, reply1) = got
        assert np.array_equal(req, req1) and np.array_equal(reply, reply1)
        bi = sched.get_batch_info(req, reply)
        n, pad = max(int(reply[0]), 0), (bi[0] + 7) // 8 * 8
        tok, pos, ctx, desc = (torch.full((k,), -7, dtype=torch.int32) for k in (pad, pad, bi[1], n * D))
        sched.get_batch_compact(req, reply, tok, pos, ctx, desc)
        host, head, lens, preempted, reqs = one.step(req1, reply1, staging)
        at = 2 * pad + (bi[1] + 3) // 4 * 4
        assert head[:4] == bi[:4] and head[4] == at + n * D + reply.size and head[10] == n
        assert lens == bi[6:] and preempted == sched.get_preempt_requests() and reqs == sched.get_batch_reqs()
        assert head[5] == (int(desc.view(n, D)[:, 3].max()) if n else 0) and head[6] == int(ctx.sum()) and head[7] == 0
        assert torch.equal(host[:2 * pad], torch.cat([tok, pos])) and torch.equal(host[2 * pad:2 * pad + bi[1]], ctx)
        assert torch.equal(host[at:at + n * D], desc) and np.array_equal(host[at + n * D:head[4]].numpy(), reply)
        alive = [r for r in alive if r not in preempted]
        last = [step] * len(alive)
        if not alive:
            break
    assert (blocks > 9) == (len(alive) == 4)
    with pytest.raises(KeyError):
        pair[1][1].step(np.array([77, 1, 0], dtype=np.int32), np.arange(1 + L * H, dtype=np.int32) * 0 + 1, staging)


def test_step_says_what_an_empty_reply_is():
    """An allocator reply without its first word is refused as get_batch_info refuses it,
    also behind a step of more than two tokens (whose count the refusal used to be looked
    up by)."""
    L, H, bs = 2, 2, 16
    store, sched = KVStorage(64 * L * H), BatchScheduler(L, H, 128, bs)
    sched.enable_device_rows(2)
    sched.add_request(np.arange(20, dtype=np.int32), 0, 8)
    buf = torch.zeros((4096,), dtype=torch.int32)
    info = sched.try_batch([0], [])
    req = np.ascontiguousarray(info[:-1])
    sched.step(req, store.allocate_batch(req, L, H), lambda n: buf)
    req = np.ascontiguousarray(sched.try_batch([0], [7])[:-1])
    with pytest.raises(ValueError):
        sched.get_batch_info(req, np.empty((0,), dtype=np.int32))
    with pytest.raises(ValueError):
        sched.step(req, np.empty((0,), dtype=np.int32), lambda n: buf)
    assert sched.step(req, np.array([1], dtype=np.int32), lambda n: buf)[1][:2] == [1, 1]


def test_staging_waits_for_the_copy_of_a_step_that_was_refused(monkeypatch):
    """The operator queues the copy out of the staging buffer before its launch can be
    refused; the next step must still wait for that copy before it packs over it."""
    from muxserve_amd import device_tables
    calls = []

    class Event:
        def record(self, stream):
            calls.append(("record", stream))

        def synchronize(self):
            calls.append(("synchronize",))

    class Operators:
        @staticmethod
        def step_inputs(*args):
            calls.append(("copy",))
            raise RuntimeError("mux_build_step: refused")

    monkeypatch.setattr(device_tables.T, "load", lambda: Operators)
    monkeypatch.setattr(torch.cuda, "Event", Event)
    monkeypatch.setattr(torch.cuda, "current_stream", lambda device: "stream")
    tables = device_tables.DeviceBlockTables(BatchScheduler(2, 2, 128, 16), 2, "cpu")
    host = tables.staging(0)
    with pytest.raises(RuntimeError):
        tables.step_inputs(host, [1, 1, 1, 1, 20, 1, 1, 0, 0, 0, 1])
    tables.staging(0)
    assert calls == [("copy",), ("record", "stream"), ("synchronize",)]
