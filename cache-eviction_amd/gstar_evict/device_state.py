"""Device state of the runtime: one object per SGLang scheduler (GPU).

It holds the tensors the reference's State holds (R:89-110; same names, shapes and dtypes, since
the hooks and tests read them) plus what this build adds: the decode score queues, cached
workspaces and the per-layer K/V pointer tables of the boundary kernels.
"""
from __future__ import annotations

import os
import threading

import torch


class State:
    """Per-row eviction state (``frontier``, ``count``, ``mode``, the shared slot ``table``), the
    per-(full layer, KV head, slot) fp32 ``scores``, the request ``entries`` by row, and the
    queued decode steps (``qq``/``qnorm``/``qlim``/``qcount`` per full layer and row; ``queued``
    mirrors the count on the host)."""

    def __init__(self, backend):
        pool = backend.token_to_kv_pool
        r2t = backend.req_to_token_pool.req_to_token
        self.pool, self.req_to_token, self.device = pool, r2t, r2t.device
        n_rows, width = r2t.shape
        # Full-attention layers in layer order; sliding-window layers keep SGLang's own cache.
        self.full_layers = [lid for lid in sorted(pool.layers_mapping) if not pool.layers_mapping[lid][1]]
        self.index = dict(zip(self.full_layers, range(len(self.full_layers))))
        self.first_full = self.full_layers[0]
        self.num_slots, self.kv_heads, self.dim = (int(x) for x in pool.get_key_buffer(self.first_full).shape)
        i32 = dict(dtype=torch.int32, device=self.device)
        self.frontier, self.count, self.mode = (torch.zeros(n_rows, **i32) for _ in range(3))
        self.table = torch.zeros((n_rows, width), **i32)
        # [layer, head, slot] view of [layer, slot, head] storage: one slot's 8 head scores are
        # adjacent, so the kernels touch a 32-byte row per slot.
        backing = torch.zeros((len(self.full_layers), self.num_slots, self.kv_heads), dtype=torch.float32,
                              device=self.device)
        self.scores = backing.permute(0, 2, 1)
        self.entries = {}
        self.verify = os.environ.get("GSTAR_EVICT_VERIFY") == "1"
        # GSTAR_EVICT_CHECK=1: the host checks every decode CSR before its launch (a debug mode:
        # it reads the CSR back, one synchronisation per call).
        self.check = os.environ.get("GSTAR_EVICT_CHECK") == "1"
        self.score_mode = os.environ.get("GSTAR_EVICT_SCORE", "queue")
        if self.score_mode not in ("queue", "eager"):
            raise ValueError("GSTAR_EVICT_SCORE must be 'queue' or 'eager'")
        self.queue_cap = int(os.environ.get("GSTAR_EVICT_QUEUE", "64"))
        if not 1 <= self.queue_cap <= 64:
            raise ValueError("GSTAR_EVICT_QUEUE must be in 1..64")
        self.q_heads = None
        self.qq = self.qnorm = self.qlim = None
        self.qcount = torch.zeros((len(self.full_layers), n_rows), **i32)
        self.queued = {}
        # Host tallies of the folds: row flushes that folded at least one queued step, and the
        # queued steps they folded (each step counts once for all full layers).
        self.folds = 0
        self.folded_steps = 0
        # The current decode step's in-launch queue folds: batch indices on the device (a slice
        # of a small ring of pinned uploads) and their count.
        self.fold_seq, self.fold_n, self.fold_wg = None, 0, 0
        self.cus = torch.cuda.get_device_properties(self.device).multi_processor_count \
            if self.device.type == "cuda" else 0
        self.fold_done = set()  # full-layer indices whose decode launch folded this step's list
        self.fold_disabled = False  # set once a decode is captured into a graph
        self._fold_ring = None
        self._fold_next = 0
        # Kept decode products (gse_score_flush_logits): row -> index in the logits buffer on the
        # device (logit_index), the rows whose products of the current step are still unfolded,
        # the full-layer indices decoded with products kept this step, and (rows, cap) of the
        # buffer's layout.
        self.logit_index = None
        self.logit_rows_on_device = {}
        self.logit_fresh = set()
        self.logit_layers = set()
        self.logit_layout = (0, 0)
        self.row_ids = torch.arange(n_rows, **i32)
        self.layer_scaling = {}  # full-layer index -> softmax scale of its queued queries
        self._ws = {}
        self._status_blocks = []  # pinned host blocks [rows, 16] of boundary status words
        self._status_blocks_used = 0
        self._pools = None
        self.pending = []  # boundaries queued on the device whose host part is still to do
        self._rows_host = self._rows_dev = self._rows_copied = None
        self._ints_host = threading.local()  # read_ints' pinned buffer, one per thread

    def workspace(self, name, nbytes):
        """A cached device byte buffer of at least nbytes (grows, never shrinks)."""
        buf = self._ws.get(name)
        if buf is None or buf.numel() < nbytes:
            # An eighth of headroom, in 2 MiB steps: a row's boundary workspace grows with its
            # candidates, and each growth is a device allocation.
            size = max(int(nbytes), 256) if buf is None else max(int(nbytes), buf.numel() + buf.numel() // 8)
            size = -(-size // (1 << 21)) << 21 if size > (1 << 21) else size
            del buf
            self._ws.pop(name, None)
            buf = self._ws[name] = torch.empty(size, dtype=torch.uint8, device=self.device)
        return buf

    def read_ints(self, *tensors):
        """The values of small integer tensors as lists, with one wait for all of them: their copies
        to the thread's pinned buffer are queued together on the current stream."""
        if any(t.device.type != "cuda" for t in tensors):
            return [t.tolist() for t in tensors]
        views, end = [], 0
        for t in tensors:
            views.append((end, end + t.numel() * t.element_size()))
            end = -(-views[-1][1] // 8) * 8
        buf = getattr(self._ints_host, "buf", None)
        if buf is None or buf.numel() < end:
            buf = self._ints_host.buf = torch.empty(max(end, 4096), dtype=torch.uint8, pin_memory=True)
        host = [buf[a:b].view(t.dtype).view(t.shape) for (a, b), t in zip(views, tensors)]
        for h, t in zip(host, tensors):
            h.copy_(t, non_blocking=True)
        torch.cuda.current_stream(self.device).synchronize()
        return [h.tolist() for h in host]

    def status_block(self, count=0):
        """A pinned host block of status rows ([rows, 16] int32, the first ``count`` for one
        boundary batch): a block of its own for every batch started since the host last finished
        all pending boundaries, so a block is not written again before its batch is finished."""
        while self._status_blocks_used >= len(self._status_blocks):
            self._status_blocks.append(torch.zeros((self.req_to_token.shape[0], 16), dtype=torch.int32,
                                                   pin_memory=True))
        block = self._status_blocks[self._status_blocks_used]
        self._status_blocks_used += 1
        return block

    def row_list(self, rows):
        """``rows`` (host ints) as a device int32 vector, through a persistent pinned buffer: the
        copy is queued on the current stream and the buffer is reused once the previous copy from
        it has completed (a multi-row flush is a few per interval, so that wait never blocks)."""
        n = len(rows)
        if self._rows_host is None:
            self._pin_rows()
        else:
            self._rows_copied.synchronize()
        self._rows_host[:n] = torch.tensor(rows, dtype=torch.int32)
        self._rows_dev[:n].copy_(self._rows_host[:n], non_blocking=True)
        self._rows_copied.record()
        return self._rows_dev[:n]

    def fold_list(self, seqs):
        """``seqs`` (host ints) as a device int32 vector for this step's decode launches, through a
        ring of four pinned uploads: a slot is written again four steps later, after waiting for
        its previous copy (long complete by then)."""
        n_rows = self.req_to_token.shape[0]
        if self._fold_ring is None:
            self._fold_ring = [(torch.zeros(n_rows, dtype=torch.int32, pin_memory=True),
                                torch.zeros(n_rows, dtype=torch.int32, device=self.device), torch.cuda.Event())
                               for _ in range(4)]
        host, dev, copied = self._fold_ring[self._fold_next]
        self._fold_next = (self._fold_next + 1) % len(self._fold_ring)
        copied.synchronize()
        n = len(seqs)
        host[:n] = torch.tensor(seqs, dtype=torch.int32)
        dev[:n].copy_(host[:n], non_blocking=True)
        copied.record()
        return dev[:n]

    def _pin_rows(self):
        if self._rows_host is None:
            total = 3 * self.req_to_token.shape[0]  # room for two row lists and one value list
            self._rows_host = torch.zeros(total, dtype=torch.int32, pin_memory=True)
            self._rows_dev = torch.zeros(total, dtype=torch.int32, device=self.device)
            self._rows_copied = torch.cuda.Event()

    def finish_pending(self):
        """Do the host part of every queued boundary, oldest first."""
        from .compaction import finish_boundary
        while self.pending:
            finish_boundary(self, self.pending.pop(0))
        self._status_blocks_used = 0  # every block's batch is finished

    def ensure_queue(self):
        """Allocate the score queues once (the decode kernels fix 8 query heads per KV head)."""
        if self.qq is not None:
            return
        n_rows, layers, cap = self.req_to_token.shape[0], len(self.full_layers), self.queue_cap
        self.q_heads = 8 * self.kv_heads
        self.qq = torch.zeros((layers, n_rows, cap, self.q_heads, self.dim), dtype=torch.bfloat16, device=self.device)
        self.qnorm = torch.zeros((layers, n_rows, cap, self.q_heads), dtype=torch.float32, device=self.device)
        self.qlim = torch.zeros((layers, n_rows, cap), dtype=torch.int32, device=self.device)
        self.logit_index = torch.full((n_rows,), -1, dtype=torch.int32, device=self.device)
        # Pinned host buffers now, at the first decode step: allocating pinned memory
        # synchronises the device, which would drain the GPU if done mid-run.
        self.status_block()
        self._status_blocks_used = 0
        self._pin_rows()

    def pool_pointers(self):
        """Device arrays of the full layers' K and V buffer addresses, and their shared strides."""
        keys = [self.pool.get_key_buffer(lid) for lid in self.full_layers]
        values = [self.pool.get_value_buffer(lid) for lid in self.full_layers]
        signature = tuple(t.data_ptr() for t in keys + values)
        if self._pools is None or self._pools[0] != signature:
            ref = keys[0]
            for t in keys + values:
                if t.dtype != torch.bfloat16 or t.stride(-1) != 1 or t.stride()[:2] != ref.stride()[:2]:
                    raise RuntimeError("gstar_evict needs bf16 K/V pools with one shared layout")
            as_table = lambda ts: torch.tensor([t.data_ptr() for t in ts], dtype=torch.int64, device=self.device)
            self._pools = (signature, as_table(keys), as_table(values), ref.stride(0), ref.stride(1))
        return self._pools[1:]

    def release_row(self, row):
        """Forget a row: its entry, policy mode, eviction state and queued decode steps (queued
        scores must not land on slots the row no longer owns)."""
        self.finish_pending()
        self.entries.pop(row, None)
        for t in (self.mode, self.frontier, self.count):
            t[row] = 0
        self.qcount[:, row] = 0
        self.queued.pop(row, None)
        self.logit_fresh.discard(row)
