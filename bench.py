#!/usr/bin/env python
"""Fused decode attention + H2O score + per-head eviction on one MI355X.

Workload: the 12 full-attention layers of gpt-oss-20b (64 query heads, 8 KV
heads, head_dim 64, bf16 K/V pool with 16-token pages), batch 32, logical
lengths uniform in [16K, 64K] (seed 2), per-KV-head budget 32768 = 512 prefix
+ 4096 recent + 28160 scored (head_sum policy), eviction every 64 tokens per
sequence, pre-compacted initial state, 2 % planted heavy-hitter keys. One step
= the CSR fill, the fused attention + score kernel of every full layer, and
every boundary (flush, select, relocate, compact) the step triggers.

Prints one JSON line. ``value`` is the whole step's algorithmic HBM traffic
divided by its time (GB/s); ``us_per_step`` is the step time.
"""
from __future__ import annotations

import argparse
import gc
import json
import math
import os
import statistics
import sys
import time
from types import SimpleNamespace

ROOT = os.path.dirname(os.path.abspath(__file__))
sys.path.insert(0, os.path.join(ROOT, "cache-eviction_amd"))
sys.path.insert(0, ROOT)

HQ, HKV, D = 64, 8, 64
PAGE = 16
PEAK_HBM_GBS = 8000.0


def parse(argv=None):
    p = argparse.ArgumentParser(description=__doc__)
    p.add_argument("--gpus", type=int, default=1)
    p.add_argument("--steps", type=int, default=512)
    p.add_argument("--warmup", type=int, default=16)
    p.add_argument("--preroll", type=int, default=-1,
                   help="untimed steps before the warm-up that bring every row's score queue to its steady-state "
                        "phase (the queue of a row at length n holds n mod interval steps); -1 = one interval")
    p.add_argument("--bs", type=int, default=32)
    p.add_argument("--layers", type=int, default=12)
    p.add_argument("--budget", type=int, default=32768)
    p.add_argument("--prefix", type=int, default=512)
    p.add_argument("--recent", type=int, default=4096)
    p.add_argument("--interval", type=int, default=64)
    p.add_argument("--min-len", type=int, default=16384)
    p.add_argument("--max-len", type=int, default=65536)
    p.add_argument("--policy", default="head_sum_2048")
    p.add_argument("--heavy", type=float, default=0.02)
    p.add_argument("--dup", type=float, default=0.0,
                   help="fraction of each layer's slots whose K row is an exact copy of another slot's")
    p.add_argument("--seed", type=int, default=2)
    p.add_argument("--ordered-pages", action="store_true",
                   help="give the rows' 16-slot pages of the pool in address order instead of shuffled (the "
                        "relocation's rate with every row's pages contiguous)")
    p.add_argument("--kernel-reps", type=int, default=20, help="launches timed per layer for the roofline")
    p.add_argument("--no-cpu-baseline", action="store_true")
    p.add_argument("--eager", action="store_true", help="score each step eagerly (second K pass per step)")
    p.add_argument("--pairs", type=int, default=200, help="off/on pairs per size and policy of --decode-latency")
    p.add_argument("--decode-latency", action="store_true",
                   help="bs=1 decode layer latency at 8K/16K/32K resident (the reference's published shape)")
    p.add_argument("--prefill-policy", default="block_sum_2048",
                   help="eviction policy of the --prefill workload (block policies: layer-shared blocks)")
    p.add_argument("--prefill-block", type=int, default=16, help="positions per block of a --prefill block policy")
    p.add_argument("--prefill-delay", type=int, default=0,
                   help="score delay of a --prefill block policy (the reference report's ARC-AGI-3 runs: 128)")
    p.add_argument("--prefill-cap", type=int, default=0,
                   help="evicted blocks per boundary of a --prefill block policy, 0 = no cap (the report: 512)")
    p.add_argument("--prefill-block-score", default="position", choices=("position", "step_max"),
                   help="block score of a --prefill block policy: accumulated position scores, or the report's "
                        "per-block counters (step maximum over a block's keys and all query heads)")
    p.add_argument("--prefill", action="store_true",
                   help="time the chunked-prefill score tiles instead: 12 layers, 79,720-token prompt in "
                        "8192-token chunks, prefix capped at the 28,672-token budget (MFMA roofline)")
    p.add_argument("--replay", action="store_true",
                   help="time static replay's layer difference instead: first full layer, 79,720-token prompt "
                        "in 2048-token chunks, 2048 positions retained per KV head (MFMA roofline)")
    p.add_argument("--reference-config", action="store_true",
                   help="run the CPU reference configuration end to end (one full layer, 4096-token prompt, boundary, "
                        "256 decode steps) on the GPU and, in fp32, on the host cores")
    p.add_argument("--copy-mib", type=int, default=0,
                   help="only run a plain device copy of this many MiB (5 launches): the byte-counter "
                        "calibration kernel for rocprofv3 FETCH_SIZE / WRITE_SIZE runs")
    return p.parse_args(argv)


def decode_bytes(n_resident):
    """Algorithmic HBM bytes of one (sequence, full layer) decode step with n resident keys.

    K and V rows (2 x 8 heads x 64 dims x 2 B), the fp32 score read + write per
    KV head, the int32 slot index; then q in and o out (64 heads x 64 dims x
    2 B each) and the 64 bf16 sinks read once per sequence.
    """
    return n_resident * (HKV * D * 2 * 2 + HKV * 4 * 2 + 4) + HQ * D * 2 * 2 + HQ * 2


def attention_bytes(n_resident):
    """Algorithmic HBM bytes of the fused attention kernel for one (sequence, layer): K and V
    rows and the slot index per key; q in, o out and the sinks. The score update is done by
    the queue flush, so its bytes are not this kernel's."""
    return n_resident * (HKV * D * 2 * 2 + 4) + HQ * D * 2 * 2 + HQ * 2


def boundary_bytes(n_cols, width, count, freed, layers):
    """Algorithmic bytes of one row's boundary: select (score + pos read, kept pos write per head)
    and compact (every kept middle K/V row and score read + written, table and leftover writes)."""
    select = layers * HKV * (n_cols * (4 + 4) + count * 4)
    move = layers * HKV * width * (2 * D * 2 * 2 + 4 * 2)
    return select + move + 4 * count + 8 * freed


def precompacted_row(n, interval, budget, prefix, recent, slots, width, middle):
    """A row of logical length n as its last boundary (at f = n - n % interval) left it, when
    f > budget: the table holds the prefix, the recent window (protected, by position) and a
    per-head sorted middle (``middle(lo, hi, count)`` draws [L, G, count] ascending positions in
    [lo, hi)); req_to_token holds the owned prefix and middle slots packed at its start, the real
    slots of the recent window [f - recent, f) and the tail [f, n) (the repack of R:485-491 with
    the cursor past the recent window). ``slots`` are the row's slots in column order: table
    columns first, then the tail. Rows with f <= budget hold positions 0..n-1 unevicted.
    Returns CPU int32 tensors: table [count], req_to_token [width], pos [L, G, count]."""
    import torch
    f = n - n % interval
    r2t = torch.zeros(width, dtype=torch.int32)
    if f <= budget:
        r2t[:n] = slots[:n].int()
        return {"frontier": 0, "count": 0, "table": None, "req_to_token": r2t, "pos": None}
    lo, hi, mid = prefix, f - recent, budget - prefix - recent
    drawn = middle(lo, hi, mid).to(torch.int32)
    layers, heads = drawn.shape[:2]
    pos = torch.empty((layers, heads, budget), dtype=torch.int32)
    pos[:, :, :prefix] = torch.arange(prefix, dtype=torch.int32)
    pos[:, :, prefix:prefix + recent] = torch.arange(hi, f, dtype=torch.int32)
    pos[:, :, prefix + recent:] = drawn
    r2t[hi:f] = slots[prefix:prefix + recent].int()
    packed = torch.cat((slots[:prefix], slots[prefix + recent:budget]))
    r2t[:packed.numel()] = packed.int()
    r2t[f:n] = slots[budget:budget + n - f].int()
    return {"frontier": f, "count": budget, "table": slots[:budget].int(), "req_to_token": r2t, "pos": pos}


def preroll_steps(args):
    """Untimed steps that bring the score queues to their steady-state phase (one interval by
    default)."""
    return args.interval if args.preroll < 0 else args.preroll


def phase_flush_rows(lens, entries, interval, budget):
    """The rows (1-based) whose score queue a pre-roll step folds itself: those at a multiple of
    the interval whose boundary there evicts nothing (count + n - frontier within the budget),
    so no boundary flushes them. A row that evicts folds its queue at each boundary (every
    ``interval`` steps, at n mod interval = 0); with these folds a row within its budget takes
    the same phase, and its queue then fills (and is flushed full) at the same point of every
    interval. After one interval of pre-roll, every row's queue holds n mod interval steps."""
    return [i + 1 for i, (n, e) in enumerate(zip(lens, entries))
            if n % interval == 0 and e["count"] + n - e["frontier"] <= budget]


def local_row_state(table_row, r2t_row, pos, count, frontier, n):
    """A row's eviction state over a local slot numbering that holds only the row's own slots:
    ``used`` (ascending global slot ids of the table and of req_to_token[:n]) maps global slot
    used[j] to local slot j + 1; local slot 0 stays the null slot. The local table and
    req_to_token are the global ones renumbered, so a boundary on them takes the same decisions
    (ownership and sliding-window checks included) as on the live row. CPU int64 tensors."""
    import torch
    table = table_row[:count].long()
    r2t = r2t_row[:n].long()
    used = torch.unique(torch.cat((table, r2t[r2t > 0])))
    local_r2t = torch.zeros(n, dtype=torch.int64)
    held = r2t > 0
    local_r2t[held] = torch.searchsorted(used, r2t[held]) + 1
    local_table = torch.searchsorted(used, table) + 1
    return {"used": used, "table": local_table, "req_to_token": local_r2t,
            "pos": None if pos is None else pos.long(), "count": count, "frontier": frontier, "n": n}


class Workload:
    """The synthetic serving state: pools, rows, eviction state, pre-drawn steps."""

    def __init__(self, args, torch, ge):
        self.args, self.torch, self.ge = args, torch, ge
        dev = torch.device("cuda")
        g = torch.Generator().manual_seed(args.seed)
        self.dgen = torch.Generator(device=dev).manual_seed(args.seed)
        bs, L, B = args.bs, args.layers, args.budget
        total_steps = preroll_steps(args) + args.warmup + args.steps
        lens = torch.randint(args.min_len, args.max_len + 1, (bs,), generator=g).tolist()
        self.lens0 = lens
        # Per-row state at the start: pre-compacted at the last interval boundary when over budget.
        rows = []
        for n in lens:
            f = n - n % args.interval
            if f > B:
                rows.append({"len": n, "frontier": f, "count": B})
            else:
                rows.append({"len": n, "frontier": 0, "count": 0})
        need = [r["count"] + (r["len"] - r["frontier"]) + total_steps + PAGE for r in rows]
        pages = [-(-x // PAGE) for x in need]
        npages = sum(pages)
        # Page-granular interleaving of rows in the pool (or each row's pages in address order).
        perm = torch.arange(npages) if args.ordered_pages else torch.randperm(npages, generator=g)
        slots = npages * PAGE + 1  # slot 0 stays the null slot
        self.slots = slots
        page_of = []
        o = 0
        for p in pages:
            page_of.append(perm[o:o + p])
            o += p
        self.row_slots = [(pp[:, None] * PAGE + torch.arange(PAGE)[None, :]).reshape(-1) + 1 for pp in page_of]
        width = max(lens) + total_steps + PAGE
        width = -(-width // 256) * 256
        # Pools: 12 full layers, random N(0, 1) bf16 with planted heavy hitters per KV head.
        keys, values = {}, {}
        self.dup_pairs = {}  # layer -> (dst, src): slot dst's key row (all heads) copied from src
        for l in range(L):
            k = torch.randn((slots, HKV, D), device=dev, dtype=torch.bfloat16)
            v = torch.randn((slots, HKV, D), device=dev, dtype=torch.bfloat16)
            gen = torch.Generator(device=dev).manual_seed(1000 + l)
            u = torch.randn((HKV, D), device=dev, generator=gen)
            u = u / u.norm(dim=-1, keepdim=True)
            nh = int(args.heavy * slots)
            for h in range(HKV):
                idx = torch.randint(1, slots, (nh,), device=dev, generator=gen)
                kk = k[idx, h].float()
                k[idx, h] = (4 * kk.norm(dim=-1, keepdim=True) * u[h]).to(torch.bfloat16)
            if args.dup > 0:
                nd = int(args.dup * slots)
                dst = torch.randperm(slots - 1, device=dev, generator=gen)[:nd] + 1
                src = torch.randint(1, slots, (nd,), device=dev, generator=gen)
                k[dst] = k[src]
                self.dup_pairs[l] = (dst, src)
            keys[l], values[l] = k, v
        pool = SimpleNamespace(layers_mapping={l: (l, False) for l in range(L)},
                               get_key_buffer=keys.__getitem__, get_value_buffer=values.__getitem__)
        self.backend = SimpleNamespace(
            token_to_kv_pool=pool, max_kv_splits=16,
            req_to_token_pool=SimpleNamespace(req_to_token=torch.zeros((bs + 1, width), dtype=torch.int32,
                                                                        device=dev)),
            kv_indptr=torch.zeros(bs + 2, dtype=torch.int32, device=dev))
        ge.STATE = None
        st = ge.state(self.backend)
        st.score_mode = "eager" if args.eager else "queue"
        self.st = st
        st.scores.uniform_(0.0, 1.0, generator=torch.Generator(device=dev).manual_seed(7))
        # A duplicated key starts with its source's scores (copied as the keys were, all sources
        # read first): the two stay exactly tied through every score update that sees both.
        for l, (dst, src) in self.dup_pairs.items():
            st.scores[l][:, dst] = st.scores[l][:, src]
        r2t = torch.zeros((bs + 1, width), dtype=torch.int32)
        table = torch.zeros((bs + 1, width), dtype=torch.int32)
        self.entries = []
        self.new_slots = []
        cfg = {"name": args.policy, "budget": B, "prefix": args.prefix, "recent": args.recent, "seed": args.seed}
        def middle(lo, hi, mid):
            draw = torch.rand((L * HKV, hi - lo), device=dev, generator=self.dgen)
            return (draw.argsort(-1)[:, :mid].sort(-1).values + lo).view(L, HKV, mid).cpu()

        for i, r in enumerate(rows):
            row = i + 1
            s = self.row_slots[i]
            e = ge._live_entry(SimpleNamespace(rid=f"r{row}", session=None), cfg, "live")
            n = r["len"]
            init = precompacted_row(n, args.interval, B, args.prefix, args.recent, s, r2t.shape[1], middle)
            f, c = init["frontier"], init["count"]
            r2t[row] = init["req_to_token"]
            if c:
                table[row, :c] = init["table"]
                e["pos"] = init["pos"].to(dev)
                e.update(frontier=f, count=c, last_boundary=f)
            else:
                e["last_boundary"] = n - n % args.interval
            nxt = s[c + n - f:]
            self.new_slots.append(nxt[:total_steps])
            st.entries[row] = e
            self.entries.append(e)
            st.mode[row] = ge.requests.score_word(e)
            st.count[row] = c
            st.frontier[row] = f
        st.req_to_token.copy_(r2t.to(dev))
        st.table.copy_(table.to(dev))
        # Each step's new slots, contiguous: int64 for out_cache_loc, int32 for req_to_token.
        self.new_slots = torch.stack(self.new_slots).t().contiguous().to(dev)  # [steps, bs]
        self.new_slots32 = self.new_slots.int()
        self.rows = torch.arange(1, bs + 1, device=dev)
        self.rows_host = list(range(1, bs + 1))
        self.lens = list(lens)
        self.seq_lens = torch.tensor(lens, dtype=torch.int64, device=dev)
        cap = sum(r["count"] + r["len"] - r["frontier"] for r in rows) + bs * (total_steps + 2)
        self.kv_indices = torch.zeros(cap, dtype=torch.int32, device=dev)
        self.q = [torch.randn((bs, HQ, D), device=dev, dtype=torch.bfloat16) for _ in range(L)]
        self.sinks = [torch.randn(HQ, device=dev, dtype=torch.bfloat16) for _ in range(L)]
        self.o = [torch.empty((bs, HQ, D), device=dev, dtype=torch.bfloat16) for _ in range(L)]
        self.layer_objs = [SimpleNamespace(sliding_window_size=-1, tp_q_head_num=HQ, tp_k_head_num=HKV,
                                           qk_head_dim=D, layer_id=l, scaling=D ** -0.5) for l in range(L)]
        self.alloc = SimpleNamespace(free_full=lambda s: None, full_to_swa_index_mapping=None)
        self.step_index = 0
        self.bytes = 0.0
        self.boundaries = 0
        self.started = []  # (sequence, n) of the boundaries queued in timed steps
        self.unaccounted = None  # sequence lengths of the last step, until its boundaries finish
        self.boundary_ms = []  # (ranking, compaction) device ms of each timed evicting boundary
        self.resident_hist = []

    def account_boundaries(self):
        """Add the algorithmic bytes of every finished boundary queued in a timed step."""
        a = self.args
        for i, n in self.started:
            ev = next(ev for ev in self.entries[i]["events"] if ev["boundary"] == n)
            if "freed" in ev:
                width = ev["after"] - (a.prefix + a.recent)
                self.bytes += boundary_bytes(ev["before"], max(width, 0), ev["after"], ev["freed"], a.layers)
                self.boundaries += 1
                self.boundary_ms.append((ev["ranking_ms"], ev["compaction_ms"]))
        self.started = []

    def resident(self, i):
        e = self.entries[i]
        return e["count"] + self.lens[i] - e["frontier"]

    def step(self, account=True, phase=False):
        """One decode step. ``phase`` (pre-roll steps): also fold the queues of the rows that
        reach a multiple of the interval without evicting, so that after one interval every row's
        queue holds n mod interval steps, as in a long-running server."""
        torch, ge, st, a = self.torch, self.ge, self.st, self.args
        # The decode hook's order (on_decode, R:692-710): finish the boundaries the previous step
        # queued, then queue the boundaries due before the new query (n tokens are cached), at
        # this workload's interval.
        ge.finish_boundaries(st)
        self.account_decode()
        due = []
        for i, e in enumerate(self.entries):
            n = self.lens[i]
            if n % a.interval == 0 and n > e["last_boundary"]:
                due.append((i + 1, e, n, n - 256))
                if account:
                    self.started.append((i, n))
        if phase:
            held = phase_flush_rows(self.lens, self.entries, a.interval, a.budget)
            if held:
                ge.flush(st, held)
        if due:
            ge._start_boundaries(st, due, self.alloc)
        # Allocate the new token's slot (SGLang's allocator), then the CSR for every full layer.
        t = self.step_index
        new = self.new_slots[t]
        st.req_to_token[self.rows, self.seq_lens] = self.new_slots32[t]
        self.seq_lens.add_(1)
        self.lens = [n + 1 for n in self.lens]
        bs = a.bs
        # Flushes rows whose score queue is full; rows due at the next step keep this step's
        # products when their queue holds only this step.
        ge.begin_decode_step(self.rows_host, st, [i + 1 for i, n in enumerate(self.lens) if n % a.interval == 0],
                             self.lens)
        ge.fill(self.backend, bs, self.seq_lens, self.rows, self.kv_indices)
        self.backend.forward_metadata = SimpleNamespace(kv_indptr=self.backend.kv_indptr[:bs + 1],
                                                        kv_indices=self.kv_indices)
        fb = SimpleNamespace(out_cache_loc=new, req_pool_indices=self.rows, seq_lens_cpu=self.max_resident_list())
        for l in range(a.layers):
            ge.decode(self.backend, self.q[l].view(bs, -1), self.layer_objs[l], fb, self.sinks[l],
                      self.o[l].view(bs, -1))
        # This step's resident counts depend on the boundaries it queued: counted once they finish.
        self.unaccounted = list(self.lens) if account else None
        self.step_index += 1

    def account_decode(self):
        """Decode bytes of the last step, from the entries as its boundaries left them."""
        if self.unaccounted is None:
            return
        res = [e["count"] + n - e["frontier"] for e, n in zip(self.entries, self.unaccounted)]
        self.resident_hist.append(sum(res) / len(res))
        self.bytes += self.args.layers * sum(decode_bytes(r) for r in res)
        self.unaccounted = None

    def finish(self):
        """Finish the queued boundaries and count what the timed steps did."""
        self.ge.finish_boundaries(self.st)
        self.account_decode()
        self.account_boundaries()

    def max_resident_list(self):
        # The split plan needs an upper bound of each row's resident count.
        return [self.resident(i) for i in range(self.args.bs)]


def kernel_roofline(w, reps):
    """Average duration of the fused decode launch (split + merge kernels) over the last step's
    inputs, with HIP events on the launch stream, and its algorithmic bytes per launch. One event
    pair brackets each pass over the layers (12 launches back to back, as in a step), so the
    average holds the launches and the gaps between them, not an event's own latency."""
    torch, ge, a = w.torch, w.ge, w.args
    bs = a.bs
    fb = SimpleNamespace(out_cache_loc=w.new_slots[max(w.step_index - 1, 0)], req_pool_indices=w.rows,
                         seq_lens_cpu=w.max_resident_list())
    # Resident counts of the last step (the CSR already in kv_indices).
    res = [w.resident(i) for i in range(bs)]
    per_launch = sum(attention_bytes(r) for r in res)
    stream = torch.cuda.current_stream()
    starts = [torch.cuda.Event(enable_timing=True) for _ in range(reps)]
    ends = [torch.cuda.Event(enable_timing=True) for _ in range(reps)]
    torch.cuda.synchronize()
    for k in range(reps):
        starts[k].record(stream)
        for l in range(a.layers):
            ge.decode(w.backend, w.q[l].view(bs, -1), w.layer_objs[l], fb, w.sinks[l], w.o[l].view(bs, -1))
        ends[k].record(stream)
    torch.cuda.synchronize()
    ms = [s.elapsed_time(e) / a.layers for s, e in zip(starts, ends)]
    avg_us = 1000 * statistics.mean(ms)
    return per_launch, avg_us


def cpu_threads():
    """Host threads for the CPU baseline: the cores this process may run on, capped by
    OMP_NUM_THREADS when the environment sets it (a host's share of its cores)."""
    cores = len(os.sched_getaffinity(0))
    cap = os.environ.get("OMP_NUM_THREADS", "")
    return min(cores, int(cap)) if cap.isdigit() and int(cap) > 0 else cores


def median_time(fn, prepare=None, repeats=5):
    """Median wall time of ``fn()`` over ``repeats`` runs after one warm-up run; ``prepare()``
    (untimed) runs before each."""
    times = []
    for k in range(repeats + 1):
        arg = prepare() if prepare is not None else None
        t0 = time.perf_counter()
        fn(arg)
        if k:
            times.append(time.perf_counter() - t0)
    return statistics.median(times)


def cpu_baseline(w, seqs=8, layers=2, repeats=5):
    """The same step on the host cores: the torch-CPU restatement (oracle/torch_cpu.py) of
    decode attention + H2O scores and of one row's boundary, on a bounded sample of this
    workload's own state, one warm-up and the median of ``repeats`` runs each, scaled to a step.

    Decode: ``seqs`` sequences spread over the resident-count range, ``layers`` layers each, at
    their real CSR lists over a local pool of the sequence's slots; scaled by resident keys to
    the batch and by layers to all full layers. Boundary: the evicting row with the most arriving
    positions, its real table / req_to_token / retained positions renumbered onto a local pool
    (``local_row_state``), on ``layers`` layers, scaled to all layers and to the measured
    boundaries per step."""
    import torch
    from oracle import torch_cpu as TC
    a, st, ge = w.args, w.st, w.ge
    torch_threads = torch.get_num_threads()
    threads = cpu_threads()
    torch.set_num_threads(threads)
    try:
        pool = w.backend.token_to_kv_pool

        def local_state(i):
            e, row, n = w.entries[i], i + 1, w.lens[i]
            return local_row_state(st.table[row].cpu(), st.req_to_token[row].cpu(),
                                   e["pos"][:layers].cpu() if e["count"] else None, e["count"], e["frontier"], n)

        def local_pools(ls):
            dev_used = ls["used"].to(st.device)
            pad = torch.zeros((1, HKV, D), dtype=torch.bfloat16)
            kp = [torch.cat((pad, pool.get_key_buffer(l)[dev_used].cpu())) for l in range(layers)]
            vp = [torch.cat((pad, pool.get_value_buffer(l)[dev_used].cpu())) for l in range(layers)]
            sc = torch.cat((torch.zeros((layers, HKV, 1)), st.scores[:layers][:, :, dev_used].cpu()), -1)
            return kp, vp, sc

        order = sorted(range(a.bs), key=w.resident)
        sample = sorted({order[round(k * (a.bs - 1) / max(seqs - 1, 1))] for k in range(seqs)})
        t_dec, keys_dec = 0.0, 0
        for i in sample:
            ls = local_state(i)
            kp, vp, sc = local_pools(ls)
            csr = torch.cat((ls["table"], ls["req_to_token"][ls["frontier"]:]))
            for l in range(layers):
                q, sinks = w.q[l][i].float().cpu(), w.sinks[l].float().cpu()
                t_dec += median_time(lambda _: TC.decode_layer(q, kp[l], vp[l], csr, sinks, D ** -0.5, sc[l]),
                                     repeats=repeats)
                keys_dec += csr.numel()
        total_keys = sum(w.resident(i) for i in range(a.bs)) * a.layers
        us_decode = 1e6 * t_dec / keys_dec * total_keys

        rows = [i for i in range(a.bs) if w.entries[i]["count"] and w.lens[i] > w.entries[i]["frontier"]]
        i = max(rows, key=lambda j: w.lens[j] - w.entries[j]["frontier"]) if rows else None
        us_boundary, candidates = 0.0, 0
        if i is not None:
            ls = local_state(i)
            kp, vp, sc = local_pools(ls)
            n = ls["n"]
            candidates = ls["count"] + n - ls["frontier"]

            def prepare():
                return ([k.clone() for k in kp], [v.clone() for v in vp], sc.clone(), ls["table"].clone(),
                        ls["req_to_token"].clone())

            def run(state):
                k, v, s, table, r2t = state
                out = TC.boundary(k, v, s, table, r2t, ls["pos"], ls["count"], ls["frontier"], n, a.budget,
                                  a.prefix, a.recent, n - 256, a.policy)
                if out is None:
                    raise RuntimeError("the sampled row did not evict")

            t_b = median_time(run, prepare, repeats)
            rate = w.boundaries / max(a.steps, 1)
            us_boundary = 1e6 * t_b * a.layers / layers * rate
    finally:
        torch.set_num_threads(torch_threads)
    return {"value": round(us_decode + us_boundary, 1), "unit": "us/step", "cores": threads, "kind": "port",
            "sample": f"torch-CPU fp32 restatement, {threads} threads, median of {repeats} after 1 warm-up: decode "
                      f"attention + head_sum scores of {len(sample)} sequences x {layers} layers ({keys_dec} keys) "
                      f"scaled by resident keys to {a.bs} sequences x {a.layers} layers "
                      f"({round(us_decode)} us); one {candidates}-candidate row boundary (selection, K/V/score "
                      f"relocation, repack) on {layers} layers scaled to {a.layers} layers x "
                      f"{w.boundaries / max(a.steps, 1):.2f} boundaries/step ({round(us_boundary)} us)"}


def measured_traffic(summary="decode_fused_kernel_bs32_32K.md"):
    """HBM bytes per launch of a workload's dominant kernel from its committed rocprofv3 summary
    (FETCH_SIZE and WRITE_SIZE of the same workload, scaled by a copy kernel's counts; the line
    ``hbm_bytes_per_launch: N``), or None."""
    path = os.path.join(ROOT, "profiles", summary)
    if not os.path.exists(path):
        return None
    for line in open(path):
        if line.startswith("hbm_bytes_per_launch:"):
            return int(line.split(":")[1])
    return None


def copy_calibration(torch, mib):
    """A plain device-to-device copy of `mib` MiB, five times, timed with events."""
    n = mib * (1 << 20)
    src = torch.randint(0, 255, (n,), dtype=torch.uint8, device="cuda")
    dst = torch.empty_like(src)
    dst.copy_(src)
    torch.cuda.synchronize()
    start, end = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
    start.record()
    for _ in range(5):
        dst.copy_(src)
    end.record()
    torch.cuda.synchronize()
    ms = start.elapsed_time(end) / 5
    print(json.dumps({"copy_bytes": n, "read_plus_write_GBs": round(2 * n / (ms * 1e-3) / 1e9, 1),
                      "avg_ms": round(ms, 4)}), flush=True)


PEAK_BF16_TFLOPS = 2500.0


class PrefillWorkload:
    """The chunked-prefill workload at the 79,720-token shape: 12 full layers of random bf16 keys
    (5 % planted heavy hitters) and values, one row whose prompt fills 79,720 slots in random
    order, one 8192-query block of random queries (each chunk takes its first ``count``), the
    row's policy config (budget 512 + 4096 + 24,064; block policies: layer-shared blocks)."""

    PROMPT, CHUNK, CAP = 79720, 8192, 512 + 4096 + 24064

    def __init__(self, args, torch, ge):
        self.args, self.torch, self.ge = args, torch, ge
        prompt, chunk = self.PROMPT, self.CHUNK
        L = self.layers = args.layers
        slots = prompt + 64
        g = torch.Generator(device="cuda").manual_seed(args.seed)
        keys, values = {}, {}
        for l in range(L):
            k = torch.randn((slots + 1, HKV, D), device="cuda", dtype=torch.bfloat16, generator=g)
            u = torch.randn((HKV, D), device="cuda", generator=g)
            u = u / u.norm(dim=-1, keepdim=True)
            heavy = torch.rand((slots + 1, HKV), device="cuda", generator=g) < 0.05
            planted = (4 * k.float().norm(dim=-1, keepdim=True) * u[None]).to(torch.bfloat16)
            keys[l] = torch.where(heavy[..., None], planted, k)
            values[l] = torch.randn((slots + 1, HKV, D), device="cuda", dtype=torch.bfloat16, generator=g)
        self.keys, self.values = keys, values
        pool = SimpleNamespace(layers_mapping={l: (l, False) for l in range(L)},
                               get_key_buffer=keys.__getitem__, get_value_buffer=values.__getitem__)
        width = -(-prompt // 256) * 256
        self.backend = SimpleNamespace(
            token_to_kv_pool=pool, max_kv_splits=16,
            req_to_token_pool=SimpleNamespace(req_to_token=torch.zeros((2, width), dtype=torch.int32, device="cuda")),
            kv_indptr=torch.zeros(3, dtype=torch.int32, device="cuda"))
        ge.STATE = None
        st = self.st = ge.state(self.backend)
        self.q = torch.randn((chunk, HQ, D), device="cuda", dtype=torch.bfloat16, generator=g)
        self.sinks = torch.randn(HQ, device="cuda", generator=g)
        st.req_to_token[1, :prompt] = (torch.randperm(slots, device="cuda", generator=g)[:prompt] + 1).int()
        self.layer_objs = [SimpleNamespace(sliding_window_size=-1, tp_q_head_num=HQ, tp_k_head_num=HKV,
                                           qk_head_dim=D, layer_id=l, scaling=D ** -0.5) for l in range(L)]
        self.cfg = {"name": args.prefill_policy, "budget": self.CAP, "prefix": 512, "recent": 4096,
                    "seed": args.seed}
        self.block_policy = args.prefill_policy in ("block_sum_2048", "block_max_2048")
        if self.block_policy:
            self.cfg.update(block=args.prefill_block, shared=True, score_delay=args.prefill_delay,
                            max_evicted_blocks=args.prefill_cap, block_score=args.prefill_block_score)
        self.starts = list(range(0, prompt, chunk))

    def run(self, timing=None, observe=None):
        """One pass over the prompt from a fresh row (no eviction state, zero scores; the pools
        keep whatever earlier passes moved): before each chunk after the first, the row's
        boundary (replay mode: survivors relocated, nothing freed); then the chunk's prefill
        scores on every layer. ``timing`` collects event pairs per chunk ("boundary", "score");
        ``observe(stage, start, entry)`` runs before ("before") and after ("after") each boundary.
        Returns the entry and the resident prefix length of each chunk."""
        torch, ge, st = self.torch, self.ge, self.st
        st.table.zero_()
        st.count.zero_()
        st.frontier.zero_()
        st.scores.zero_()
        entry = ge._live_entry(SimpleNamespace(rid="prompt", session=None), self.cfg, "replay")
        if entry["error"]:
            raise ValueError(f"--prefill config: {entry['error']}")
        st.entries[1] = entry
        word = ge.requests.score_word(entry)  # score mode and delay
        st.mode[1] = word
        resident = []
        for start in self.starts:
            count = min(self.CHUNK, self.PROMPT - start)
            ev = [torch.cuda.Event(enable_timing=True) for _ in range(3)]
            ev[0].record()
            if start:
                if observe:
                    observe("before", start, entry)
                ge._boundary(st, 1, entry, start)
                if observe:
                    observe("after", start, entry)
            ev[1].record()
            prefix = torch.cat((st.table[1, :entry["count"]], st.req_to_token[1, entry["frontier"]:start]))
            new = st.req_to_token[1, start:start + count]
            for l in range(self.layers):
                ge._prefill_scores(st, l, word, self.layer_objs[l], self.q[:count], self.keys[l], self.sinks,
                                   prefix, new)
            ev[2].record()
            resident.append(prefix.numel())
            if timing is not None:
                timing["boundary"].append(ev[:2])
                timing["score"].append(ev[1:])
        return entry, resident


def prefill_bench(args, torch, ge):
    """Chunked prefill at the 79,720-token shape with eviction: one row prefills 8192-token
    chunks; before each chunk the row's boundary keeps 512 + 4096 + 24,064 positions with the
    block policy (16-token blocks chosen per layer, one choice for all KV heads, block score =
    the sum of its positions' scores; ``--prefill-policy`` picks another), then per chunk and
    layer the exact causal softmax probabilities (sink in the normaliser) over the row's
    resident keys are summed per KV head onto the keys' scores.
    Scoring work = 2 * 64 heads * 64 dims flop per causal (query, key) pair for one QK^T pass
    (the kernel issues a second pass: the normaliser first, then the probabilities). Boundaries
    run in replay mode (survivors relocated, nothing freed) and are timed separately."""
    w = PrefillWorkload(args, torch, ge)
    prompt, chunk, cap, L, starts = w.PROMPT, w.CHUNK, w.CAP, w.layers, w.starts
    block_policy = w.block_policy
    timing = {"score": [], "boundary": []}

    w.run()
    torch.cuda.synchronize()
    start, end = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
    reps = max(1, min(args.steps, 3))  # one step is the whole 79,720-token prompt (about a second)
    start.record()
    for _ in range(reps):
        entry, resident = w.run(timing)
    end.record()
    torch.cuda.synchronize()
    ms = start.elapsed_time(end) / reps
    score_ms = sum(a.elapsed_time(b) for a, b in timing["score"]) / reps
    boundary_ms = sum(a.elapsed_time(b) for a, b in timing["boundary"]) / reps
    pairs = sum(r * min(chunk, prompt - s) + min(chunk, prompt - s) * (min(chunk, prompt - s) + 1) // 2
                for r, s in zip(resident, starts))
    flop = L * pairs * 2 * HQ * D
    tflops = flop / (score_ms * 1e-3) / 1e12
    evictions = [ev for ev in entry["events"] if "freed" in ev]
    baseline = None
    if not args.no_cpu_baseline:
        try:
            baseline = cpu_prefill_baseline(w, resident, starts, pairs * L)
        except Exception as problem:  # noqa: BLE001
            import traceback
            traceback.print_exc()
            baseline = {"value": None, "unit": "TFLOP/s", "error": repr(problem)}
    # Relocation bytes per evicting boundary: every head's kept middle K+V row read and written
    # and its score read and written (the width is the budget minus the 4608 protected).
    moved = sum(L * HKV * (ev["after"] - 4608) * (2 * 2 * D * 2 + 4 * 2) for ev in evictions)
    policy = args.prefill_policy.replace("_2048", "")
    if block_policy:
        policy += f" {args.prefill_block}-token layer-shared blocks"
        policy += f", score delay {args.prefill_delay}" if args.prefill_delay else ""
        policy += f", at most {args.prefill_cap} blocks evicted per boundary" if args.prefill_cap else ""
        if args.prefill_block_score == "step_max":
            policy += ", per-block counters (step maximum over a block's keys and all query heads)"
    return {
        "metric": "chunked-prefill score tiles, TFLOP/s (one QK^T pass) and % of bf16 MFMA peak",
        "value": round(tflops, 1), "unit": "TFLOP/s", "n_gpus": 1, "steps": reps, "warmup": 1,
        "ms_per_step": round(ms, 3), "higher_is_better": True, "scaling": "weak", "vs_baseline": None,
        "dtype": "bf16", "data": "synthetic",
        "config": {"workload": f"gpt-oss-20b chunked prefill, {L} layers, 79,720-token prompt in 8192-token chunks, "
                               f"{policy}, budget {cap} "
                               f"(512+4096+24064), 5% heavy-hitter keys",
                   "causal_pairs_per_layer": pairs},
        "roofline": {"bound": "mfma", "achieved": round(tflops, 1), "peak": PEAK_BF16_TFLOPS, "unit": "TFLOP/s",
                     "frac": round(tflops / PEAK_BF16_TFLOPS, 4), "issued_frac": round(2 * tflops / PEAK_BF16_TFLOPS, 4),
                     # HBM bytes per (chunk, layer) of the score launches, from the committed profile of the
                     # default --prefill workload.
                     "traffic": measured_traffic("prefill_kernel_79720.md") if prefill_default(args) else None},
        "cpu_baseline": baseline,
        # Two exponentials per (query head, key) pair (normaliser pass, probability pass).
        "exp2_T_per_s": round(2 * L * pairs * HQ / (score_ms * 1e-3) / 1e12, 2),
        "score_ms": round(score_ms, 3),
        "eviction": {"policy": args.prefill_policy, "boundaries": len(evictions),
                     "evicted_per_boundary": [ev["before"] - ev["after"] for ev in evictions],
                     "boundary_ms": round(boundary_ms, 3),
                     # The last run's relocated bytes over one run's boundary time (selection, block
                     # scores, relocation and the host wait included).
                     "relocation_GB_s": round(moved / (boundary_ms * 1e-3) / 1e9, 1) if boundary_ms else None},
    }


def prefill_default(args):
    """True for the --prefill workload the committed profile covers (the default policy flags)."""
    return (args.prefill_policy, args.prefill_block, args.prefill_delay, args.prefill_cap,
            args.prefill_block_score, args.layers) == ("block_sum_2048", 16, 0, 0, "position", 12)


def cpu_prefill_baseline(w, resident, starts, total_pairs, sample=2048):
    """The prefill scores on the host cores: the torch-CPU restatement (oracle/torch_cpu.py) of
    R:314-340 for the last ``sample`` queries of a full 8192-query chunk of the workload at its
    largest resident prefix (each over every earlier key of the chunk and the whole prefix), on
    one layer (the workload's own keys, queries and sinks, random slot order), after a 64-query
    warm-up; extrapolated by causal (query, key) pairs to the whole prompt on every layer and
    reported as the same one-pass TFLOP/s as the GPU line."""
    import torch
    from oracle import torch_cpu as TC
    chunk = w.CHUNK
    full = [(r, s) for r, s in zip(resident, starts) if min(chunk, w.PROMPT - s) == chunk]
    prefix_len, _ = max(full)
    first = chunk - sample  # the sampled queries are the chunk's last
    threads = cpu_threads()
    torch_threads = torch.get_num_threads()
    torch.set_num_threads(threads)
    try:
        keys = w.keys[0].cpu()
        q = w.q[first:chunk].cpu()
        sinks = w.sinks.float().cpu()
        g = torch.Generator().manual_seed(1)
        slots = torch.randperm(keys.shape[0] - 1, generator=g)[:prefix_len + chunk] + 1
        scores = torch.zeros((HKV, keys.shape[0]))
        TC.prefill_scores(q[:64], keys, slots[:prefix_len + first + 64], prefix_len + first, sinks, D ** -0.5, scores)
        t0 = time.perf_counter()
        TC.prefill_scores(q, keys, slots, prefix_len + first, sinks, D ** -0.5, scores)
        seconds = time.perf_counter() - t0
    finally:
        torch.set_num_threads(torch_threads)
    pairs = (prefix_len + first) * sample + sample * (sample + 1) // 2
    prompt_s = seconds * total_pairs / pairs
    return {"value": round(pairs * 2 * HQ * D / seconds / 1e12, 3), "unit": "TFLOP/s", "cores": threads,
            "kind": "port", "repeats": 1,
            "sample": f"torch-CPU fp32 restatement of R:314-340, {threads} threads: the last {sample} queries of an "
                      f"{chunk}-query chunk over its {prefix_len}-key resident prefix on one layer ({pairs} causal "
                      f"pairs) in {seconds:.2f} s after a 64-query warm-up; extrapolated by causal pairs to the whole "
                      f"prompt on {w.layers} layers: {prompt_s:.1f} s per prompt"}


def decode_latency_bench(args, torch, ge):
    """One full-attention decode layer at bs=1 (64 q heads, 8 KV heads, d=64, bf16, 16-token pages
    in random order), at 8192, 16384 and 32768 resident keys: the shape of the reference's own
    published timings (SGLang decode attention alone, then with its score kernel). Per size, with
    HIP events over 200 calls replayed from HIP graphs of 32 calls (after 20 warmups):
      attention  - a row without a score policy (mode 0): attention only;
      queued     - head_sum: attention, the step queued, plus the flush of a full 64-step queue
                   for this layer amortised over its 64 steps (timed separately);
      eager      - head_sum with the score added in the same call (a second pass over K).
    Then, per size and policy (head_sum, head_max_sum), the reference's paired off/on protocol
    (``paired_timing``, TM:58-87): per-call event pairs, launch path included."""
    dev = torch.device("cuda")
    g = torch.Generator(device=dev).manual_seed(args.seed)
    sizes = (2048, 8192, 16384, 32768)
    slots = max(sizes) + 64
    k = torch.randn((slots + 1, HKV, D), device=dev, dtype=torch.bfloat16, generator=g)
    v = torch.randn((slots + 1, HKV, D), device=dev, dtype=torch.bfloat16, generator=g)
    pool = SimpleNamespace(layers_mapping={0: (0, False)}, get_key_buffer=lambda l: k, get_value_buffer=lambda l: v)
    width = slots + 256
    backend = SimpleNamespace(token_to_kv_pool=pool, max_kv_splits=8,
                              req_to_token_pool=SimpleNamespace(req_to_token=torch.zeros((2, width), dtype=torch.int32,
                                                                                         device=dev)),
                              kv_indptr=torch.zeros(3, dtype=torch.int32, device=dev))
    pages = torch.randperm(slots // PAGE, device=dev, generator=g)
    order = (pages[:, None] * PAGE + torch.arange(PAGE, device=dev)[None]).reshape(-1) + 1
    q = torch.randn((1, HQ, D), device=dev, dtype=torch.bfloat16, generator=g)
    sinks = torch.randn(HQ, device=dev, dtype=torch.bfloat16, generator=g)
    o = torch.empty((1, HQ, D), device=dev, dtype=torch.bfloat16)
    lay = SimpleNamespace(sliding_window_size=-1, tp_q_head_num=HQ, tp_k_head_num=HKV, qk_head_dim=D, layer_id=0,
                          scaling=D ** -0.5)
    rows = torch.tensor([1], device=dev)
    reps, warm = 200, 20

    def timed(fn, n):
        """Per-call µs of ``fn`` replayed from a HIP graph of 32 calls (the GPU's time, without the
        Python launch path, which is slower than a bs=1 layer)."""
        for _ in range(warm):
            fn()
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            for _ in range(32):
                fn()
        graph.replay()
        torch.cuda.synchronize()
        start, end = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        replays = max(1, n // 32)
        start.record()
        for _ in range(replays):
            graph.replay()
        end.record()
        torch.cuda.synchronize()
        return 1000 * start.elapsed_time(end) / (replays * 32)

    results = []
    for n in sizes:
        out = {"resident": n}
        for mode_name, score_mode, policy_mode in (("attention", "queue", 0), ("queued", "queue", 1),
                                                     ("eager", "eager", 1)):
            ge.STATE = None
            st = ge.state(backend)
            st.score_mode = score_mode
            st.mode[1] = policy_mode
            st.req_to_token[1, :n] = order[:n].int()
            kv_indices = torch.zeros(n, dtype=torch.int32, device=dev)
            ge.fill(backend, 1, torch.tensor([n], device=dev), rows, kv_indices)
            backend.forward_metadata = SimpleNamespace(kv_indptr=backend.kv_indptr[:2], kv_indices=kv_indices)
            fb = SimpleNamespace(out_cache_loc=order[n - 1:n], req_pool_indices=rows, seq_lens_cpu=[n])

            def step():
                # Past the queue's capacity the merge only counts the step (no entry is written):
                # the queue's flush is timed below.
                ge.decode(backend, q.view(1, -1), lay, fb, sinks, o.view(1, -1))

            us = timed(step, reps)
            if mode_name == "queued":
                # A full queue: 64 steps of this layer, then one flush (the step loop above reset it).
                st.qcount.fill_(st.queue_cap)
                st.qlim[:, 1] = n
                st.qnorm[:, 1] = 10.0
                st.qq[:, 1] = q.view(1, 1, HQ, D).expand(-1, st.queue_cap, -1, -1)

                def flush():
                    st.qcount[:, 1] = st.queue_cap
                    st.queued[1] = st.queue_cap
                    ge.flush(st, [1])

                flush_us = timed(flush, 20)
                out["queued_flush_us"] = round(flush_us, 1)
                us += flush_us / st.queue_cap
            out[f"{mode_name}_us"] = round(us, 2)
        out["attention_GB_s"] = round((2052 * n + 16512) / (out["attention_us"] * 1e-6) / 1e9, 1)
        out["paired"] = [paired_timing(torch, ge, backend, mode, q, lay, sinks, o, order, n, policy, args, queued)
                         for queued in (False, True) for policy, mode in (("head_sum_2048", 1), ("head_max_sum_2048", 2))]
        results.append(out)
    baseline = None
    if not args.no_cpu_baseline:
        # The same layer on the host cores: the torch-CPU restatement (attention + head_sum
        # scores, R:155-224), median of 5 after a warm-up, per size.
        from oracle import torch_cpu as TC
        threads = cpu_threads()
        torch_threads = torch.get_num_threads()
        torch.set_num_threads(threads)
        try:
            kc, vc, qc, sc = k.cpu(), v.cpu(), q[0].float().cpu(), sinks.float().cpu()
            cpu_us = {}
            for n in sizes:
                slots = order[:n].cpu()
                scores = torch.zeros((HKV, kc.shape[0]))
                cpu_us[str(n)] = round(1e6 * median_time(lambda _: TC.decode_layer(qc, kc, vc, slots, sc, D ** -0.5,
                                                                                    scores)), 1)
        finally:
            torch.set_num_threads(torch_threads)
        for out in results:
            out["cpu_us"] = cpu_us[str(out["resident"])]
        baseline = {"value": cpu_us[str(sizes[1])], "unit": "us", "cores": threads, "kind": "port", "repeats": 5,
                    "per_size_us": cpu_us,
                    "sample": f"torch-CPU fp32 restatement of one decode layer (attention with sinks + head_sum scores, "
                              f"R:155-224), bs=1, {threads} threads, median of 5 after a warm-up, at every size; value at "
                              f"{sizes[1]} resident (the line's value size)"}
    return {
        "metric": "bs=1 decode layer latency (gpt-oss-20b full-attention shape), us",
        "value": results[1]["queued_us"], "unit": "us", "n_gpus": 1, "steps": reps, "warmup": warm,
        "higher_is_better": False, "scaling": "weak", "vs_baseline": None, "dtype": "bf16", "data": "synthetic",
        "config": {"workload": "one full-attention decode layer, bs=1, 64 q heads, 8 KV heads, d=64, bf16, "
                               "16-token pages in random order, head_sum, resident 2048 / 8192 / 16384 / 32768 "
                               "(value: 8192)"},
        "sizes": results,
        "cpu_baseline": baseline,
        "reference_gb10": {"8192": {"attention_us": 58.9, "with_scores_us": 83.9},
                           "16384": {"attention_us": 150.0, "with_scores_us": 192.9}},
    }


def paired_timing(torch, ge, backend, mode, q, lay, sinks, o, order, n, policy, args, queued=False):
    """The reference's paired protocol (TM:58-87) on one full-attention layer at bs=1: "off" is
    the decode attention alone, "on" the same call with the policy's score update added before
    it returns (the reference's per-step `after_decode`). Eager path: the second pass over K.
    Queued path (the default): the decode step as the runtime runs it, begin_decode_step and
    the decode inside the timed call, so an "on" sample queues the step and one in 64 also
    folds the full queue (the flush runs in the step that finds the queue full). Each sample is
    one call between two events with a synchronize on each side, the scores are zeroed outside
    the timed region (eager), pairs alternate their order, and 20 warm-up pairs run first.
    Reports the means, the paired deltas and the overhead."""
    import statistics
    dev = q.device
    ge.STATE = None
    st = ge.state(backend)
    st.score_mode = "queue" if queued else "eager"
    rows = torch.tensor([1], device=dev)
    st.req_to_token[1, :n] = order[:n].int()
    kv_indices = torch.zeros(n, dtype=torch.int32, device=dev)
    ge.fill(backend, 1, torch.tensor([n], device=dev), rows, kv_indices)
    backend.forward_metadata = SimpleNamespace(kv_indptr=backend.kv_indptr[:2], kv_indices=kv_indices)
    fb = SimpleNamespace(out_cache_loc=order[n - 1:n], req_pool_indices=rows, seq_lens_cpu=[n])
    start, end = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)

    def timed(on):
        st.mode[1] = mode if on else 0
        if on:
            st.entries[1] = {"mode": mode}  # the host's view of the row's score kind
        else:
            st.entries.pop(1, None)
        if not queued:
            st.scores.zero_()
        torch.cuda.synchronize()
        start.record()
        if queued:
            ge.begin_decode_step([1], st)
        ge.decode(backend, q.view(1, -1), lay, fb, sinks, o.view(1, -1))
        end.record()
        torch.cuda.synchronize()
        return start.elapsed_time(end)

    for _ in range(20):
        timed(False), timed(True)
    pairs = []
    for i in range(args.pairs):
        order_i = (False, True) if i % 2 == 0 else (True, False)
        sample = {on: timed(on) for on in order_i}
        pairs.append((sample[False], sample[True]))
    deltas = [b - a for a, b in pairs]
    off, on = statistics.mean(a for a, _ in pairs), statistics.mean(b for _, b in pairs)
    st.entries.pop(1, None)
    return {"policy": policy, "path": "queued" if queued else "eager", "pairs": len(pairs), "warmup_pairs": 20,
            "synchronization": "hip_event_per_sample",
            "off_us": round(1000 * off, 2), "on_us": round(1000 * on, 2), "extra_us": round(1000 * (on - off), 2),
            "paired_delta_mean_us": round(1000 * statistics.mean(deltas), 2),
            "paired_delta_stdev_us": round(1000 * statistics.stdev(deltas), 2),
            "overhead_percent": round(100 * (on - off) / off, 1)}


def replay_bench(args, torch, ge):
    """Static replay's layer difference over a 79,720-token prompt in 2048-token chunks with
    2048 positions retained per KV head after each boundary: per chunk, the first full layer's
    output over every earlier key and over each head's survivors, then the per-query relative
    error. Algorithmic work = 4 * 64 dims flop per (query head, visible key) pair and output
    (QK^T and PV, one each); the kernel issues PV twice (probabilities as bf16 hi + lo)."""
    prompt, chunk, budget = 79720, 2048, 2048
    g = torch.Generator(device="cuda").manual_seed(args.seed)
    k = torch.randn((prompt, HKV, D), device="cuda", generator=g)
    u = torch.randn((HKV, D), device="cuda", generator=g)
    heavy = torch.rand((prompt, HKV), device="cuda", generator=g) < 0.02
    k = torch.where(heavy[..., None], 4 * k.norm(dim=-1, keepdim=True) * (u / u.norm(dim=-1, keepdim=True)), k)
    sk = k.to(torch.bfloat16)
    sv = torch.randn((prompt, HKV, D), device="cuda", generator=g).to(torch.bfloat16)
    q = torch.randn((chunk, HQ, D), device="cuda", generator=g).to(torch.bfloat16)
    sinks = torch.randn(HQ, device="cuda", generator=g)
    layer = SimpleNamespace(tp_q_head_num=HQ, tp_k_head_num=HKV, qk_head_dim=D, scaling=D ** -0.5)
    pool = SimpleNamespace(layers_mapping={0: (0, False)}, get_key_buffer=lambda l: sk, get_value_buffer=lambda l: sv)
    backend = SimpleNamespace(token_to_kv_pool=pool, max_kv_splits=16,
                              req_to_token_pool=SimpleNamespace(req_to_token=torch.zeros((2, 64), dtype=torch.int32,
                                                                                         device="cuda")),
                              kv_indptr=torch.zeros(3, dtype=torch.int32, device="cuda"))
    ge.STATE = None
    st = ge.state(backend)
    plan = []  # (start, count, entry): the boundary at each multiple of 2048 above the budget evicts
    for start in range(0, prompt, chunk):
        count = min(chunk, prompt - start)
        entry = {"shadow_k": sk, "shadow_v": sv, "frontier": 0, "count": 0, "layer_error": []}
        if start > budget:
            pos = torch.rand((HKV, start), device="cuda", generator=g).argsort(-1)[:, :budget].sort(-1).values
            entry.update(frontier=start, count=budget, pos=pos.to(torch.int32)[None])
        plan.append((start, count, entry))

    def run():
        for start, count, entry in plan:
            entry["layer_error"].clear()
            ge._replay_layer_difference(st, entry, q[:count], layer, sinks, start)

    run()
    torch.cuda.synchronize()
    t0, t1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
    reps = max(1, min(args.steps, 5))
    t0.record()
    for _ in range(reps):
        run()
    t1.record()
    torch.cuda.synchronize()
    ms = t0.elapsed_time(t1) / reps
    pairs = sum(start * count + count * (count + 1) // 2 for start, count, _ in plan)
    kept_pairs = sum(budget * count + count * (count + 1) // 2 for start, count, e in plan if e["count"])
    flop = (pairs + kept_pairs) * HQ * 4 * D
    tflops = flop / (ms * 1e-3) / 1e12
    baseline = None
    if not args.no_cpu_baseline:
        try:
            baseline = cpu_replay_baseline(plan[-1], q, sk, sv, sinks, budget, flop)
        except Exception as problem:  # noqa: BLE001
            import traceback
            traceback.print_exc()
            baseline = {"value": None, "unit": "TFLOP/s", "error": repr(problem)}
    return {
        "metric": "replay layer difference, TFLOP/s (QK^T + PV per output) and % of bf16 MFMA peak",
        "value": round(tflops, 1), "unit": "TFLOP/s", "n_gpus": 1, "steps": reps, "warmup": 1,
        "ms_per_step": round(ms, 3), "higher_is_better": True, "scaling": "weak", "vs_baseline": None,
        "dtype": "bf16", "data": "synthetic",
        "config": {"workload": "gpt-oss-20b first full layer, 79,720-token prompt in 2048-token chunks, 2048 "
                               "positions retained per KV head, 2% heavy-hitter keys",
                   "causal_pairs": pairs, "retained_pairs": kept_pairs},
        "roofline": {"bound": "mfma", "achieved": round(tflops, 1), "peak": PEAK_BF16_TFLOPS, "unit": "TFLOP/s",
                     "frac": round(tflops / PEAK_BF16_TFLOPS, 4), "issued_frac": round(1.5 * tflops / PEAK_BF16_TFLOPS, 4),
                     "traffic": None},
        "exp2_T_per_s": round((pairs + kept_pairs) * HQ / (ms * 1e-3) / 1e12, 2),
        "cpu_baseline": baseline,
    }


def cpu_replay_baseline(last, q, sk, sv, sinks, budget, total_flop, sample=128):
    """The replay layer difference on the host cores: the torch-CPU restatement (oracle/torch_cpu.py)
    of R:520-546 for the first ``sample`` queries of the prompt's last chunk (its real retained
    positions; the longest key range), after a 16-query warm-up; its algorithmic work (QK^T and
    PV over every earlier key and over the visible ones) scaled to the whole prompt."""
    import torch
    from oracle import torch_cpu as TC
    start, count, entry = last
    n = min(sample, count)
    end = start + n
    visible = torch.zeros((HKV, end), dtype=torch.bool)
    visible[:, entry["frontier"]:] = True
    visible.scatter_(1, entry["pos"][0].long().cpu(), True)
    threads = cpu_threads()
    torch_threads = torch.get_num_threads()
    torch.set_num_threads(threads)
    try:
        qc, skc, svc, sc = q[:n].cpu(), sk[:end].cpu(), sv[:end].cpu(), sinks.float().cpu()
        TC.replay_errors(qc[:16], skc[:start + 16], svc[:start + 16], sc, D ** -0.5, visible, start)
        t0 = time.perf_counter()
        TC.replay_errors(qc, skc, svc, sc, D ** -0.5, visible, start)
        seconds = time.perf_counter() - t0
    finally:
        torch.set_num_threads(torch_threads)
    flop = sum((start + i + 1) + (budget + i + 1) for i in range(n)) * HQ * 4 * D
    return {"value": round(flop / seconds / 1e12, 3), "unit": "TFLOP/s", "cores": threads, "kind": "port",
            "repeats": 1,
            "sample": f"torch-CPU fp32 restatement of R:520-546, {threads} threads: the first {n} queries of the last "
                      f"chunk (positions {start}..{end - 1}, {int(visible.sum())} visible (head, position) entries) in "
                      f"{seconds:.2f} s after a 16-query warm-up, same algorithmic flop count as the GPU line; "
                      f"extrapolated: {seconds * total_flop / flop:.1f} s per prompt"}


def reference_config_bench(args, torch, ge):
    """The CPU reference configuration end to end, on the GPU and on the host cores: one
    full-attention layer of gpt-oss-20b shape, a 4096-token prompt in two 2048-token chunks
    (prefill scores, R:314-340), the boundary at 4096 before the first decode query (head_sum,
    budget 2048 = 128 prefix + 512 recent + 1408 scored, R:415-491), then 256 decode steps
    (attention with sinks and the H2O score, R:155-224). Q, K, V ~ N(0, 1) and the sinks from
    seed 0, scale 1/8. The GPU runs its bf16 kernels (K, V and Q in bf16) through the runtime's
    hooks, one decode launch per step (launch-bound at this size); the CPU baseline runs the
    torch-CPU restatement in fp32, as the configuration states. value: GPU ms for the whole flow;
    also the retained positions' overlap between the two (exact up to near-ties: bf16 vs fp32)."""
    from oracle import torch_cpu as TC
    prompt, chunk, steps = 4096, 2048, 256
    budget, prefix, recent = 2048, 128, 512
    total = prompt + steps
    g = torch.Generator().manual_seed(0)
    Q = torch.randn((total, HQ, D), generator=g)
    K = torch.randn((total, HKV, D), generator=g)
    V = torch.randn((total, HKV, D), generator=g)
    sinks = torch.randn(HQ, generator=g)
    scale = D ** -0.5
    dev = torch.device("cuda")
    # Slot p + 1 holds position p; slot 0 is the null slot.
    kp = torch.zeros((total + 1, HKV, D), dtype=torch.bfloat16, device=dev)
    vp = torch.zeros_like(kp)
    kp[1:], vp[1:] = K.to(torch.bfloat16).to(dev), V.to(torch.bfloat16).to(dev)
    qd, sd = Q.to(torch.bfloat16).to(dev), sinks.to(dev)
    pool = SimpleNamespace(layers_mapping={0: (0, False)}, get_key_buffer=lambda l: kp, get_value_buffer=lambda l: vp)
    backend = SimpleNamespace(token_to_kv_pool=pool, max_kv_splits=16, kv_indptr=torch.zeros(3, dtype=torch.int32, device=dev),
                              req_to_token_pool=SimpleNamespace(req_to_token=torch.zeros((2, total + 64), dtype=torch.int32,
                                                                                         device=dev)))
    lay = SimpleNamespace(sliding_window_size=-1, tp_q_head_num=HQ, tp_k_head_num=HKV, qk_head_dim=D, layer_id=0,
                          scaling=scale)
    cfg = {"name": "head_sum_2048", "budget": budget, "prefix": prefix, "recent": recent, "seed": 0}
    alloc = SimpleNamespace(free_full=lambda s: None, full_to_swa_index_mapping=None)
    rows = torch.tensor([1], device=dev)
    kv_indices = torch.zeros(total + 64, dtype=torch.int32, device=dev)
    o = torch.empty((1, HQ, D), dtype=torch.bfloat16, device=dev)

    def gpu_run():
        ge.STATE = None
        st = ge.state(backend)
        st.req_to_token[1, :total] = torch.arange(1, total + 1, dtype=torch.int32, device=dev)
        e = ge._live_entry(SimpleNamespace(rid="reference", session=None), cfg, "live")
        st.entries[1] = e
        word = ge.requests.score_word(e)
        st.mode[1] = word
        for start in range(0, prompt, chunk):
            if start:
                ge._boundary(st, 1, e, start, None, alloc)  # 2048 resident: within the budget, an event
            resident = torch.cat((st.table[1, :e["count"]], st.req_to_token[1, e["frontier"]:start]))
            ge._prefill_scores(st, 0, word, lay, qd[start:start + chunk], kp, sd, resident,
                               st.req_to_token[1, start:start + chunk])
        for t in range(steps):
            n = prompt + t
            if n % chunk == 0 and n > e["last_boundary"]:
                ge._boundary(st, 1, e, n, None, alloc)
            ge.begin_decode_step([1], st, [], [n + 1])
            seq = torch.tensor([n + 1], device=dev)
            ge.fill(backend, 1, seq, rows, kv_indices)
            backend.forward_metadata = SimpleNamespace(kv_indptr=backend.kv_indptr[:2], kv_indices=kv_indices)
            fb = SimpleNamespace(out_cache_loc=seq.clone(), req_pool_indices=rows,
                                 seq_lens_cpu=[e["count"] + n + 1 - e["frontier"]])
            ge.decode(backend, qd[n].view(1, -1), lay, fb, sd, o.view(1, -1))
        ge.flush(st)
        return e

    gpu_run()
    torch.cuda.synchronize()
    reps = max(1, min(args.steps, 5))
    times = []
    for _ in range(reps):
        torch.cuda.synchronize()
        t0 = time.perf_counter()
        entry = gpu_run()
        torch.cuda.synchronize()
        times.append(time.perf_counter() - t0)
    gpu_ms = 1000 * statistics.median(times)

    def cpu_run():
        kp32, vp32 = torch.cat((torch.zeros(1, HKV, D), K)), torch.cat((torch.zeros(1, HKV, D), V))
        scores = torch.zeros((1, HKV, total + 1))
        for start in range(0, prompt, chunk):
            TC.prefill_scores(Q[start:start + chunk], kp32, torch.arange(1, start + chunk + 1), start, sinks, scale,
                              scores[0])
        table = torch.zeros(total + 64, dtype=torch.int64)
        r2t = torch.zeros(total + 64, dtype=torch.int64)
        r2t[:total] = torch.arange(1, total + 1)
        count, pos, _ = TC.boundary([kp32], [vp32], scores, table, r2t, None, 0, 0, prompt, budget, prefix, recent)
        for t in range(steps):
            n = prompt + t
            scores[:, :, n + 1] = 0.0
            slots = torch.cat((table[:count], r2t[prompt:n + 1]))
            TC.decode_layer(Q[n], kp32, vp32, slots, sinks, scale, scores[0])
        return pos

    threads = cpu_threads()
    torch_threads = torch.get_num_threads()
    torch.set_num_threads(threads)
    try:
        cpu_pos = cpu_run()
        cpu_s = median_time(lambda _: cpu_run(), repeats=3)
    finally:
        torch.set_num_threads(torch_threads)
    gpu_pos = entry["pos"][0].long().cpu()
    overlap = sum(len(set(gpu_pos[h].tolist()) & set(cpu_pos[0, h].tolist())) for h in range(HKV)) / (HKV * budget)
    return {
        "metric": "CPU reference configuration end to end (one full layer: 4096-token prompt, boundary, 256 decode "
                  "steps), ms",
        "value": round(gpu_ms, 2), "unit": "ms", "n_gpus": 1, "steps": reps, "warmup": 1, "ms_per_step": round(gpu_ms, 3),
        "higher_is_better": False, "scaling": "weak", "vs_baseline": None, "dtype": "bf16", "data": "synthetic",
        "config": {"workload": "one gpt-oss-20b full-attention layer (64 q heads, 8 KV heads, d=64), batch 1, "
                               "4096-token prompt in two 2048-token chunks then 256 decode steps, head_sum budget 2048 "
                               "(128 + 512 + 1408), boundary at 4096, Q/K/V/sinks ~ N(0,1) seed 0"},
        "retained_overlap_vs_cpu_fp32": round(overlap, 4),
        "cpu_baseline": {"value": round(1000 * cpu_s, 2), "unit": "ms", "cores": threads, "kind": "port", "repeats": 3,
                         "sample": f"the whole configuration in fp32 with the torch-CPU restatement (prefill scores "
                                   f"R:314-340, boundary R:415-491, 256 decode steps R:155-224), {threads} threads, "
                                   f"median of 3 after a warm-up"},
    }


def workload_name(args):
    k = lambda n: f"{n // 1024}K" if n % 1024 == 0 else str(n)
    scored = args.budget - args.prefix - args.recent
    name = (f"gpt-oss-20b full-attention decode, {args.layers} layers, bs={args.bs}, lengths "
            f"U[{k(args.min_len)},{k(args.max_len)}], budget {args.budget} ({args.prefix}+{args.recent}+{scored}), "
            f"{args.policy.replace('_2048', '')}, evict every {args.interval} step{'s' if args.interval > 1 else ''}, "
            f"16-token pages{' in address order' if args.ordered_pages else ''}, {args.heavy * 100:g}% heavy hitters")
    if args.dup:
        name += f", {args.dup * 100:g}% duplicate keys"
    return name


def main():
    args = parse()
    if args.gpus != 1:
        print(json.dumps({"error": "this build runs on one GPU; multi-GPU sharding is design-only",
                          "n_gpus": args.gpus}))
        sys.exit(2)
    import torch
    import gstar_evict as ge
    if not torch.cuda.is_available():
        print(json.dumps({"error": "no GPU visible"}))
        sys.exit(1)
    if args.copy_mib:
        copy_calibration(torch, args.copy_mib)
        return
    if args.prefill:
        print(json.dumps(prefill_bench(args, torch, ge)), flush=True)
        return
    if args.replay:
        print(json.dumps(replay_bench(args, torch, ge)), flush=True)
        return
    if args.decode_latency:
        print(json.dumps(decode_latency_bench(args, torch, ge)), flush=True)
        return
    if args.reference_config:
        print(json.dumps(reference_config_bench(args, torch, ge)), flush=True)
        return
    w = Workload(args, torch, ge)
    for _ in range(preroll_steps(args)):
        w.step(account=False, phase=True)
    for _ in range(args.warmup):
        w.step(account=False)
    ge.finish_boundaries(w.st)
    torch.cuda.synchronize()
    # The objects made so far (the workload's setup) leave the collector's scans: a full
    # collection over them stalled one timed step by 30 ms (measured at the eviction-at-every-step
    # shape), which is the Python heap's cost, not the path's.
    gc.collect()
    gc.freeze()
    start, end = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
    folds0, folded0 = w.st.folds, w.st.folded_steps
    t0 = time.perf_counter()
    start.record()
    for _ in range(args.steps):
        w.step(account=True)
    w.finish()
    end.record()
    torch.cuda.synchronize()
    wall = time.perf_counter() - t0
    gpu_ms = start.elapsed_time(end)
    ms_step = gpu_ms / args.steps
    gbs = w.bytes / (gpu_ms / 1000) / 1e9
    per_launch, avg_us = kernel_roofline(w, args.kernel_reps)
    achieved = per_launch / (avg_us * 1e-6) / 1e9
    # The committed counter summary covers the default workload only.
    traffic = measured_traffic() if workload_name(args) == workload_name(parse([])) else None
    result = {
        "metric": "fused attn+score+evict µs/decode-step & HBM GB/s (% peak), bs=32, 32K budget",
        "value": round(gbs, 1), "unit": "GB/s", "n_gpus": 1, "steps": args.steps, "warmup": args.warmup,
        "ms_per_step": round(ms_step, 4), "us_per_step": round(1000 * ms_step, 1), "higher_is_better": True,
        "scaling": "weak", "vs_baseline": None, "dtype": "bf16", "data": "synthetic",
        "config": {"workload": workload_name(args),
                   "batch": args.bs, "layers": args.layers, "budget": args.budget, "interval": args.interval,
                   "policy": args.policy, "score_mode": "eager" if args.eager else "queue",
                   "mean_resident": round(statistics.mean(w.resident_hist), 1),
                   "boundaries": w.boundaries, "wall_s": round(wall, 3),
                   "preroll_steps": preroll_steps(args),
                   "queue_phase": "steady: each row's score queue holds n mod interval steps at the first timed step",
                   # Queued decode steps folded into the scores inside the timed region, per step:
                   # about bs at the steady state (each step queues one per row, folded once).
                   "folds": w.st.folds - folds0,
                   "folded_steps_per_step": round((w.st.folded_steps - folded0) / args.steps, 2)},
        "roofline": {"bound": "hbm", "kernel": f"decode_fused_kernel+decode_merge_kernel (one layer, bs={args.bs})",
                     "achieved": round(achieved, 1), "peak": PEAK_HBM_GBS, "unit": "GB/s",
                     "frac": round(achieved / PEAK_HBM_GBS, 4), "traffic": traffic,
                     "bytes_per_launch": per_launch, "avg_launch_us": round(avg_us, 2)},
        "step_frac_of_peak": round(gbs / PEAK_HBM_GBS, 4),
        # Medians over the timed evicting boundaries, device time from the boundary's events:
        # ranking = score flush + selection + relocation, compaction = leftover scores, repack.
        "boundary_median_ms": {
            "ranking": round(statistics.median(r for r, _ in w.boundary_ms), 3) if w.boundary_ms else None,
            "compaction": round(statistics.median(c for _, c in w.boundary_ms), 3) if w.boundary_ms else None},
        # Everything a step adds to its decode attention (score flush, selection, compaction, CSR
        # fill, host waits), relative to the attention launches alone.
        "evict_overhead_vs_attention": round((1000 * ms_step - args.layers * avg_us) / (args.layers * avg_us), 4),
    }
    if not args.no_cpu_baseline:
        # The GPU measurement is complete here: a failure of the host-side baseline is reported in
        # its field, never allowed to lose the line.
        try:
            result["cpu_baseline"] = cpu_baseline(w)
        except Exception as problem:  # noqa: BLE001
            import traceback
            traceback.print_exc()
            result["cpu_baseline"] = {"value": None, "unit": "us/step", "error": repr(problem)}
    print(json.dumps(result), flush=True)


if __name__ == "__main__":
    main()
