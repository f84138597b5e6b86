"""Device-resident mirror of the requests' block-id runs and the step-input
builder on top of it.

The reference rebuilds the whole block table and one slot per (token, layer,
head) on the host every step and uploads them
(csrc/batch_scheduler.cpp:131-169, muxserve/flexserver/llm_runtime.py:301-327).
With a DeviceBlockTables attached to a BatchScheduler a step uploads only the
token ids, positions, context lengths, the allocator's reply and 8 ints per
sequence - in one copy - and `mux_build_step` derives slot_mapping and the
step's block table on the device, bit-identical to the reference path's.
"""
from typing import Tuple

import torch

from . import torch_ops as T
from .batch_scheduler import BatchScheduler


class DeviceBlockTables:
    def __init__(self, scheduler: BatchScheduler, max_rows: int, device="cuda:0"):
        self.scheduler = scheduler
        self.device = torch.device(device)
        self.max_rows = int(max_rows)
        self.L, self.H = scheduler.num_layers, scheduler.num_heads
        self.block_size = scheduler.block_size
        self.max_blocks_per_seq = scheduler.max_blocks_per_seq
        # int32 [row][token block][layer][head]; written only by step_inputs().
        self.mirror = torch.zeros((self.max_rows, self.max_blocks_per_seq, self.L, self.H), dtype=torch.int32,
                                  device=self.device)
        self._staging = None
        self._uploaded = None
        scheduler.enable_device_rows(self.max_rows)

    def staging(self, n_ints: int) -> torch.Tensor:
        """Grow-only pinned int32 buffer the step's upload is packed into.  The
        previous step's copy out of it must have run before it is overwritten."""
        if self._uploaded is not None:
            self._uploaded.synchronize()
        if self._staging is None or self._staging.numel() < n_ints:
            self._staging = torch.empty((max(n_ints, 1 << 16),), dtype=torch.int32,
                                        pin_memory=torch.cuda.is_available())
        return self._staging

    def step_inputs(self, host: torch.Tensor, head) -> Tuple[torch.Tensor, ...]:
        """host, head: the packed step and its sizes from BatchScheduler.step.  One
        asynchronous copy and one launch; returns token ids and positions int64
        [padded], context lens int32 on the device and on the host (a tensor of its own:
        the staging buffer is reused by the next step), slot_mapping int64 [tokens, L, H]
        and block_tables int32 [L, sequences, H, max blocks], or the reference's empty
        prefill table."""
        operator = T.load().step_inputs
        try:
            return operator(self.mirror, host, head, self.block_size)
        finally:
            # (also of a step that was refused: its copy may have been queued before that)
            if self._uploaded is None:
                self._uploaded = torch.cuda.Event()
            self._uploaded.record(torch.cuda.current_stream(self.device))
