"""Timed cases of the eviction runtime: the work its users have it do, through the hooks they call.

All at the gpt-oss-20b full-attention shape the kernels serve (64 query heads, 8 KV heads, head_dim
64, bf16 K/V in 16-token pages in random page order). The kinds:

  step        one decode step of all full layers from a captured HIP graph (CSR fill, every layer's
              fused attention with its queued scores), as a server replays it: ``on_decode`` before
              the step, which folds the score queues when they are full
  decode      one full layer's ``decode`` hook called eagerly, the queues folding in the launches
  lse         one layer's ``after_decode`` hook: scores from an external attention's split LSEs
  prefill     one layer's ``after_extend`` hook of one prefill chunk: column sums or maxima
  counters    the same for a block policy with per-step block counters and a score delay
  diagnose    the same for a regret diagnostic of several policies
  replay      the same for static replay: every query's error of the first full layer
  boundary    ``on_decode`` at a row's eviction boundary and the host part after it

Lengths, budgets and chunk sizes are those of the repository's workloads: budgets 2K to 32K, lengths
up to 64K, batches of 1 to 32, chunks of 2048 tokens (the size the runtime's boundaries ask for) and
of 8192, the last chunk of a prompt of any size.
"""
import math
import os
import random
import sys
from types import SimpleNamespace

import torch

_PKG = os.path.join(os.getcwd(), "cache-eviction_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

import gstar_evict as ge  # noqa: E402

HQ, HKV, D = 64, 8, 64
GROUP = HQ // HKV
PAGE = 16
INTERVAL = 2048
CONTEXT = 131072  # req_to_token's width: the model's context length
SPLITS, MIN_BLOCK_KV = 16, 32  # an external decode kernel's split layout
SCALE = D ** -0.5


def listed():
    return [
        # A single request at the smallest budget: the launches and their latency are the step.
        dict(name="step_bs1_2k", kind="step", bs=1, lo=4300, hi=4300, budget=2048, layers=12, policy="head_sum_2048"),
        # A single request at the largest budget.
        dict(name="step_bs1_32k", kind="step", bs=1, lo=45000, hi=45000, budget=32768, layers=12,
             policy="head_sum_2048"),
        # A small ragged batch at a middle budget, maxima instead of sums.
        dict(name="step_bs8_8k", kind="step", bs=8, lo=3000, hi=24000, budget=8192, layers=12,
             policy="head_max_sum_2048"),
        # The main serving workload's layer: 32 ragged requests of 16K to 64K tokens at a 32K budget.
        dict(name="decode_bs32_32k", kind="decode", bs=32, lo=16384, hi=65536, budget=32768, policy="head_sum_2048"),
        # A server that keeps its own attention kernel and hands over its log-sum-exps.
        dict(name="after_decode_bs8_16k", kind="lse", bs=8, lo=4000, hi=40000, budget=16384, policy="head_sum_2048"),
        # The first chunk of a prompt.
        dict(name="prefill_2k_first", kind="prefill", chunk=2048, prefix=0, policy="head_sum_2048"),
        # The last, short chunk of a long prompt.
        dict(name="prefill_1896_after_30k", kind="prefill", chunk=1896, prefix=30720, policy="head_max_sum_2048"),
        # A large chunk of the long-prompt workload, its prefix at the budget.
        dict(name="prefill_8k_after_28k", kind="prefill", chunk=8192, prefix=28672, policy="head_sum_2048"),
        # Block eviction with per-step counters: blocks of 4 tokens, counted 128 tokens late.
        dict(name="counters_2k_after_12k", kind="counters", chunk=2048, prefix=12288, block=4, delay=128),
        # The regret diagnostic of four policies, a chunk in the middle of a prompt.
        dict(name="diagnose_2k_at_14k", kind="diagnose", chunk=2048, prefix=14336, specs=4),
        # Static replay of a chunk in the middle of a prompt, 2048 positions kept per head.
        dict(name="replay_2k_at_16k", kind="replay", chunk=2048, prefix=16384, budget=2048),
        # One request's eviction at the largest budget, all layers.
        dict(name="boundary_32k", kind="boundary", budget=32768, prefix=512, recent=4096, layers=12, n=49152),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """A case of one of the kinds, its sizes spread over the kind's range."""
    kind = rng.choice(("step", "step", "decode", "lse", "prefill", "prefill", "counters", "diagnose", "replay",
                       "boundary"))
    policy = rng.choice(("head_sum_2048", "head_max_sum_2048"))
    if kind in ("step", "decode", "lse"):
        bs = _log(rng, 1, 8 if kind == "step" else 32)
        hi = _log(rng, 300, 65536)
        c = dict(kind=kind, bs=bs, lo=rng.randint(max(40, hi // 4), hi), hi=hi, budget=_log(rng, 2048, 32768),
                 policy=policy)
        return dict(c, layers=12) if kind == "step" else c
    if kind == "boundary":
        budget = rng.randrange(1, 17) * INTERVAL
        n = budget + rng.randrange(1, 9) * INTERVAL
        return dict(kind=kind, budget=budget, prefix=rng.choice((128, 512)), recent=budget // 8, layers=12, n=n)
    chunk = 2048 if rng.random() < 0.4 else _log(rng, 17, 2047)
    prefix = rng.randrange(0, 15) * INTERVAL
    if kind == "prefill":
        if rng.random() < 0.25:
            chunk = rng.randint(2049, 8192)
        # After an eviction a prefix is of any length.
        return dict(kind=kind, chunk=chunk, prefix=_log(rng, 1, 28672) if rng.random() < 0.7 else prefix,
                    policy=policy)
    if kind == "counters":
        return dict(kind=kind, chunk=chunk, prefix=prefix, block=rng.choice((4, 16)), delay=rng.choice((0, 128)))
    if kind == "diagnose":
        return dict(kind=kind, chunk=chunk, prefix=prefix // 2 // INTERVAL * INTERVAL, specs=rng.randint(1, 6))
    return dict(kind=kind, chunk=chunk, prefix=prefix, budget=rng.randrange(1, 4) * INTERVAL)


# Inputs ---------------------------------------------------------------------------------------

def _rows(case):
    """(length, frontier, count) of each request of a batch: past its budget a request holds
    ``budget`` positions of what lies before its last boundary, and everything since."""
    r = random.Random(case["bs"] * 1000003 + case["hi"])
    rows = []
    for _ in range(case["bs"]):
        n = r.randint(case["lo"], case["hi"])
        n += (n + 1) % INTERVAL < 2  # not at a boundary, nor one step before it
        n += (n + 1) % INTERVAL < 2
        f = n - n % INTERVAL
        rows.append((n, f, case["budget"]) if f > case["budget"] else (n, 0, 0))
    return rows


def _resident(case):
    return [count + n - f for n, f, count in _rows(case)]


def _generator(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _randn(g, *shape):
    return torch.randn(shape, generator=g, device="cuda", dtype=torch.bfloat16)


def _keys(g, slots):
    """N(0, 1) keys, 2 % of them heavy hitters along a direction of their head."""
    k = _randn(g, slots, HKV, D)
    u = torch.randn((HKV, D), generator=g, device="cuda")
    heavy = torch.rand((slots, HKV, 1), generator=g, device="cuda") < 0.02
    planted = 4 * k.float().norm(dim=-1, keepdim=True) * (u / u.norm(dim=-1, keepdim=True))
    return torch.where(heavy, planted.to(torch.bfloat16), k)


def _paged(g, entries):
    """``entries`` slots (never slot 0) in 16-token pages, the pages in random order; the pool's size."""
    pages = -(-entries // PAGE)
    order = torch.randperm(pages, generator=g, device="cuda")
    slots = (order[:, None] * PAGE + torch.arange(PAGE, device="cuda")).reshape(-1) + 1
    return slots[:entries].int(), pages * PAGE + 1


def _decode_inputs(case, seed):
    """A decode batch's pools, lists, queries and sinks."""
    g = _generator(seed)
    lens = _resident(case)
    starts = [0]
    for n in lens:
        starts.append(starts[-1] + -(-n // PAGE) * PAGE)  # a page belongs to one request
    slots, size = _paged(g, starts[-1])
    layers = case.get("layers", 1)
    x = SimpleNamespace(lists=[slots[s:s + n] for s, n in zip(starts, lens)], size=size, layers=layers)
    x.k = [_keys(g, size) for _ in range(layers)]
    x.v = [_randn(g, size, HKV, D) for _ in range(layers)]
    x.q = [_randn(g, len(lens), HQ, D) for _ in range(layers)]
    x.sinks = [_randn(g, HQ) for _ in range(layers)]
    if case["kind"] == "lse":
        x.splits = torch.full((len(lens),), SPLITS, dtype=torch.int32, device="cuda")
        x.lse = torch.stack([_split_lse(x.q[0][b], x.k[0][lst.long()]) for b, lst in enumerate(x.lists)])
    return x


def _split_lse(q, keys):
    """[heads, splits] log-sum-exps of one sequence's logits in the external kernel's split layout."""
    n = keys.shape[0]
    per = -(-(-(-n // SPLITS)) // MIN_BLOCK_KV) * MIN_BLOCK_KV
    logits = torch.matmul(q.float().view(HKV, GROUP, D), keys.float().permute(1, 2, 0).contiguous()) * SCALE
    out = torch.zeros((HQ, SPLITS), device="cuda")
    for s in range(-(-n // per)):
        out[:, s] = torch.logsumexp(logits[..., s * per:(s + 1) * per], -1).reshape(HQ)
    return out


def _chunk_inputs(case, seed):
    """A prefill chunk's pool, slots, queries and sinks."""
    g = _generator(seed)
    slots, size = _paged(g, case["prefix"] + case["chunk"])
    x = SimpleNamespace(slots=slots, size=size, k=_keys(g, size), v=_randn(g, size, HKV, D))
    x.q, x.sinks = _randn(g, case["chunk"], HQ, D), _randn(g, HQ)
    start = case["prefix"]
    if case["kind"] == "replay" and start > case["budget"]:
        x.kept = torch.rand((HKV, start), generator=g, device="cuda").argsort(-1)[:, :case["budget"]].sort(-1).values
    if case["kind"] == "diagnose":
        # Each policy holds half of the positions before the last boundary, other ones per head.
        x.resident = torch.ones((case["specs"], 1, HKV, start + case["chunk"]), dtype=torch.bool, device="cuda")
        if start:
            x.resident[..., :start] = torch.rand((case["specs"], 1, HKV, start), generator=g, device="cuda") < 0.5
    return x


# The runtime around them ------------------------------------------------------------------------

def _backend(k, v, rows):
    pool = SimpleNamespace(layers_mapping={l: (l, False) for l in range(len(k))}, get_key_buffer=k.__getitem__,
                           get_value_buffer=v.__getitem__)
    table = torch.zeros((rows + 1, CONTEXT), dtype=torch.int32, device="cuda")
    return SimpleNamespace(token_to_kv_pool=pool, max_kv_splits=SPLITS,
                           req_to_token_pool=SimpleNamespace(req_to_token=table),
                           kv_indptr=torch.zeros(rows + 2, dtype=torch.int32, device="cuda"))


def _runtime(backend):
    ge.STATE = None
    return ge.state(backend)


def _layer(index):
    return SimpleNamespace(sliding_window_size=-1, tp_q_head_num=HQ, tp_k_head_num=HKV, qk_head_dim=D,
                           layer_id=index, scaling=SCALE)


def _entry(name, kind, budget=2048, prefix=128, recent=512, **more):
    cfg = dict(name=name, budget=budget, prefix=prefix, recent=recent, seed=0, **more)
    entry = ge._live_entry(SimpleNamespace(rid="r", session=None), cfg, kind)
    assert not entry["error"], entry["error"]
    return entry


def _prepare_decode(case, seed):
    x = _decode_inputs(case, seed)
    bs, rows = case["bs"], _rows(case)
    lens = [n for n, _, _ in rows]
    b = _backend(x.k, x.v, bs)
    st = _runtime(b)
    s = SimpleNamespace(kind=case["kind"], x=x, b=b, st=st, lens=lens, ids=list(range(1, bs + 1)), graph=None)
    for row, (n, f, count), lst in zip(s.ids, rows, x.lists):
        entry = st.entries[row] = _entry(case["policy"], "live", case["budget"], 128, 512)
        entry.update(frontier=f, count=count, last_boundary=f)
        st.frontier[row], st.count[row], st.mode[row] = f, count, entry["mode"]
        st.table[row, :count] = lst[:count]
        st.req_to_token[row, f:n] = lst[count:]
    s.rows = torch.tensor(s.ids, device="cuda")
    s.seq_lens = torch.tensor(lens, device="cuda")
    s.o = torch.zeros((x.layers, bs, HQ * D), dtype=torch.bfloat16, device="cuda")
    s.q = [q.view(bs, HQ * D) for q in x.q]
    s.layer = [_layer(l) for l in range(x.layers)]
    s.indices = torch.zeros(sum(_resident(case)) + PAGE, dtype=torch.int32, device="cuda")
    s.fb = SimpleNamespace(out_cache_loc=torch.stack([lst[-1] for lst in x.lists]).long(), req_pool_indices=s.rows,
                           seq_lens_cpu=torch.tensor(lens))
    s.batch = SimpleNamespace(reqs=[SimpleNamespace(rid="r", session=None, kv=SimpleNamespace(req_pool_idx=r))
                                    for r in s.ids], seq_lens_cpu=s.fb.seq_lens_cpu)
    ge.fill(b, bs, s.seq_lens, s.rows, s.indices)
    b.forward_metadata = SimpleNamespace(kv_indptr=b.kv_indptr[:bs + 1], kv_indices=s.indices)
    if case["kind"] == "lse":
        b.forward_metadata.attn_lse, b.forward_metadata.num_kv_splits = x.lse, x.splits
    elif case["kind"] == "step":
        _decode_layers(s)  # the queues and workspaces are there before the capture
        torch.cuda.synchronize()
        st.qcount.zero_()
        torch.cuda.synchronize()
        s.graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(s.graph):
            ge.fill(b, bs, s.seq_lens, s.rows, s.indices)
            _decode_layers(s)
    else:
        # One queue's worth of steps, each request's queue emptied at a step of its own: requests
        # of a server do not come to their boundaries together.
        for i in range(st.queue_cap):
            _eager_step(s)
            ge.flush(st, [r for r in s.ids if r * st.queue_cap // (bs + 1) == i])
        st.scores.zero_()
    return s


def _decode_layers(s):
    for l, layer in enumerate(s.layer):
        ge.decode(s.b, s.q[l], layer, s.fb, s.x.sinks[l], s.o[l])


def _eager_step(s):
    ge.begin_decode_step(s.ids, s.st, (), s.lens)
    _decode_layers(s)


def _prepare_chunk(case, seed):
    x = _chunk_inputs(case, seed)
    kind, count, start = case["kind"], case["chunk"], case["prefix"]
    b = _backend([x.k], [x.v], 1)
    st = _runtime(b)
    if kind == "diagnose":
        req = SimpleNamespace(rid="r", session=None, origin_input_ids=range(start + count))
        specs = ",".join(f"{('head_sum_2048', 'head_max_sum_2048', 'random_2048')[j % 3]}:{max(2048, start // 2)}"
                         f":128:512" for j in range(case["specs"]))
        entry = ge._diagnostic_entry(req, {"policies": specs, "seed": 0}, st.device, 1, HKV)
        entry.update(resident=x.resident, frontier=start)
    elif kind == "counters":
        entry = _entry("block_max_2048", "live", block=case["block"], shared=True, score_delay=case["delay"],
                       block_score="step_max")
    elif kind == "replay":
        entry = _entry("random_reservoir_2048", "replay", case["budget"])
        ge._shadow(st, entry, start + count)
        entry["shadow_k"][:start], entry["shadow_v"][:start] = x.k[x.slots[:start].long()], x.v[x.slots[:start].long()]
        if start > case["budget"]:
            entry.update(count=case["budget"], frontier=start, pos=x.kept.int()[None])
    else:
        entry = _entry(case["policy"], "live")
    st.entries[1] = entry
    s = SimpleNamespace(kind=kind, x=x, b=b, st=st, entry=entry, layer=_layer(0), q=x.q.view(count, HQ * D))
    bounds = lambda n: torch.tensor([0, n], dtype=torch.int32, device="cuda")
    b.forward_metadata = SimpleNamespace(qo_indptr=bounds(count), kv_indptr=bounds(start), kv_indices=x.slots[:start])
    s.fb = SimpleNamespace(req_pool_indices=torch.tensor([1], device="cuda"), out_cache_loc=x.slots[start:].long(),
                           extend_prefix_lens_cpu=[start])
    return s


def _prepare_boundary(case, seed):
    """A row one boundary after its last one: ``budget`` kept positions and an interval of new
    ones, with positions, scores and slots as the last boundary and the decoding since left them."""
    g = _generator(seed)
    budget, n, layers = case["budget"], case["n"], case["layers"]
    f = n - INTERVAL
    evicted = f > budget
    count, frontier = (budget, f) if evicted else (0, 0)
    candidates = count + n - frontier
    slots, size = _paged(g, candidates)
    k = [_randn(g, size, HKV, D) for _ in range(layers)]
    v = [_randn(g, size, HKV, D) for _ in range(layers)]
    b = _backend(k, v, 1)
    st = _runtime(b)
    entry = st.entries[1] = _entry("head_sum_2048", "live", budget, case["prefix"], case["recent"])
    r2t = torch.zeros(CONTEXT, dtype=torch.int32, device="cuda")
    pos = None
    if evicted:
        lo, hi = case["prefix"], f - case["recent"]
        middle = budget - case["prefix"] - case["recent"]
        drawn = torch.rand((layers * HKV, hi - lo), generator=g, device="cuda").argsort(-1)[:, :middle]
        drawn = (drawn.sort(-1).values + lo).view(layers, HKV, middle)
        fixed = torch.cat((torch.arange(lo, device="cuda"), torch.arange(hi, f, device="cuda")))
        pos = torch.cat((fixed.expand(layers, HKV, -1), drawn), -1).int()
        packed = torch.cat((slots[:lo], slots[lo + case["recent"]:budget]))
        r2t[hi:f], r2t[:packed.numel()] = slots[lo:lo + case["recent"]], packed
    r2t[frontier:n] = slots[count:]
    # Accumulated attention: heavy-tailed, more for older tokens than for the newest.
    scores = torch.rand((layers, size, HKV), generator=g, device="cuda").pow_(4).permute(0, 2, 1)
    mapping = torch.zeros(size, dtype=torch.int64, device="cuda")
    freed = []
    allocator = SimpleNamespace(free_full=freed.append, full_to_swa_index_mapping=mapping)
    req = SimpleNamespace(rid="r", session=None,
                          kv=SimpleNamespace(req_pool_idx=1, get_evicted_seqlen=lambda kind: n - 128))
    batch = SimpleNamespace(reqs=[req], seq_lens_cpu=torch.tensor([n]),
                            tree_cache=SimpleNamespace(token_to_kv_pool_allocator=allocator))
    row = torch.zeros(CONTEXT, dtype=torch.int32, device="cuda")
    row[:count] = slots[:count]
    return SimpleNamespace(kind="boundary", k=k, v=v, st=st, entry=entry, batch=batch, freed=freed, n=n, pos=pos,
                           count=count, frontier=frontier, row=row, r2t=r2t, scores=scores)


def prepare(case, seed):
    if case["kind"] == "boundary":
        return _prepare_boundary(case, seed)
    return (_prepare_decode if case["kind"] in ("step", "decode", "lse") else _prepare_chunk)(case, seed)


# One pass ---------------------------------------------------------------------------------------

def run(s):
    ge.STATE = s.st
    if s.kind == "step":
        ge.on_decode(s.batch)
        s.graph.replay()
        return {"o": s.o, "norm": s.st.qnorm}
    if s.kind == "decode":
        _eager_step(s)
        return {"o": s.o, "scores": s.st.scores}
    if s.kind == "lse":
        ge.after_decode(s.b, s.q[0], s.layer[0], s.fb, s.x.sinks[0])
        return {"scores": s.st.scores}
    if s.kind == "boundary":
        return _run_boundary(s)
    if s.kind == "replay":
        s.entry["layer_error"].clear()
    ge.after_extend(s.b, s.q, s.layer, s.fb, s.x.sinks)
    if s.kind == "diagnose":
        return {name: s.entry[name] for name in ("score_sum", "score_max", "lost")}
    return {"error": s.entry["layer_error"][0]} if s.kind == "replay" else {"scores": s.st.scores}


def _run_boundary(s):
    """The row as decoding left it (its lists and scores; the K and V of earlier passes stay
    where those moved them), then its boundary."""
    st, e = s.st, s.entry
    st.table[1], st.req_to_token[1] = s.row, s.r2t
    st.count[1:2].fill_(s.count), st.frontier[1:2].fill_(s.frontier)
    st.scores.copy_(s.scores)
    e.update(count=s.count, frontier=s.frontier, last_boundary=0, pos=s.pos)
    e["events"].clear(), s.freed.clear()
    ge.on_decode(s.batch)
    ge.finish_boundaries()
    return {"pos": e["pos"], "table": st.table[1], "req_to_token": st.req_to_token[1], "freed": s.freed[0],
            "scores": st.scores, "k": s.k, "v": s.v}


# What a pass cannot do without ------------------------------------------------------------------

def _pairs(count, start):
    return count * start + count * (count + 1) // 2


def work(case):
    kind = case["kind"]
    if kind in ("step", "decode", "lse"):
        keys, bs = sum(_resident(case)), case["bs"]
        if kind == "lse":  # K, the slot list and the scores, read and written
            return {"bytes": keys * (HKV * D * 2 + 4 + HKV * 8) + bs * HQ * D * 2, "flops": keys * HQ * D * 2}
        layers = case.get("layers", 1)  # K, V and the list; q and o
        return {"bytes": layers * (keys * (HKV * D * 4 + 4) + bs * HQ * D * 4),
                "flops": layers * keys * HQ * D * 4}
    if kind == "boundary":
        n, budget, heads = case["n"], case["budget"], case["layers"] * HKV
        candidates = budget + INTERVAL if n - INTERVAL > budget else n
        middle = budget - case["prefix"] - case["recent"]
        select = heads * (candidates * 8 + budget * 4)
        return {"bytes": select + heads * middle * (2 * D * 2 * 2 + 8), "flops": 0}
    count, start = case["chunk"], case["prefix"]
    total = start + count
    pairs = _pairs(count, start)
    read = count * HQ * D * 2 + total * (HKV * D * 2 + 4)
    if kind == "replay":
        if start > case["budget"]:
            pairs += _pairs(count, case["budget"])
        return {"bytes": read + total * HKV * D * 2, "flops": pairs * HQ * D * 4}
    scores = total * HKV * 8 * (2 if kind == "diagnose" else 1)
    return {"bytes": read + (total * 8 if kind == "counters" else scores), "flops": pairs * HQ * D * 2}


def tolerance(case):
    return {
        # bf16 outputs (and probabilities rounded to bf16 before the value product); normalisers
        # and scores are 32-bit sums of exponentials of bf16 products.
        "step": {"rel": 8e-3, "max": 0.1}, "decode": {"rel": 8e-3, "max": 0.1},
        "lse": {"rel": 1e-5, "max": 1e-3}, "prefill": {"rel": 1e-5, "max": 1e-3},
        "counters": {"rel": 1e-5, "max": 1e-3}, "diagnose": {"rel": 1e-5, "max": 1e-3},
        "replay": {"rel": 1e-5, "max": 1e-3},
        "boundary": "exact",  # the kept set is a rank of given scores; everything else is moved
    }[case["kind"]]


# The same in 64 bits ------------------------------------------------------------------------------

def exact(case, seed):
    if case["kind"] == "boundary":
        return None
    return (_exact_decode if case["kind"] in ("step", "decode", "lse") else _exact_chunk)(case, seed)


def _exact_decode(case, seed):
    x = _decode_inputs(case, seed)
    bs = case["bs"]
    o = torch.zeros((x.layers, bs, HQ * D), dtype=torch.float64, device="cuda")
    norms = torch.zeros((x.layers, bs + 1, 64, HQ), dtype=torch.float64, device="cuda")
    scores = torch.zeros((1, HKV, x.size), dtype=torch.float64, device="cuda")
    for l in range(x.layers):
        for b, lst in enumerate(x.lists):
            at = lst.long()
            q, k = x.q[l][b].double().view(HKV, GROUP, D), x.k[l][at].double().permute(1, 2, 0).contiguous()
            logits = torch.matmul(q, k) * SCALE
            sink = x.sinks[l].double()
            if case["kind"] == "lse":
                per = -(-(-(-len(lst) // SPLITS)) // MIN_BLOCK_KV) * MIN_BLOCK_KV
                inner = torch.logsumexp(x.lse[b, :, :-(-len(lst) // per)].double(), -1)
            else:
                inner = torch.logsumexp(logits, -1).reshape(HQ)
            norm = torch.logaddexp(inner, sink)
            p = torch.exp(logits - norm.view(HKV, GROUP, 1))
            if case["kind"] == "lse":
                scores[0, :, at] = p.sum(1) if case["policy"] == "head_sum_2048" else p.amax(1)
            else:
                o[l, b] = torch.matmul(p, x.v[l][at].double().transpose(0, 1).contiguous()).reshape(-1)
                norms[l, b + 1, 0] = norm
    if case["kind"] == "lse":
        return {"scores": scores}
    return {"o": o, "norm": norms} if case["kind"] == "step" else {"o": o, "scores": None}


def _exact_chunk(case, seed):
    x = _chunk_inputs(case, seed)
    kind, count, start = case["kind"], case["chunk"], case["prefix"]
    total = start + count
    if _pairs(count, start) > 1.2e8:
        return None
    at = x.slots.long()
    keys, values = x.k[at].double(), x.v[at].double()
    step = max(1, min(count, (1 << 26) // (HQ * total)))
    place = torch.arange(total, device="cuda")
    f64 = dict(dtype=torch.float64, device="cuda")
    sums, maxes = torch.zeros((HKV, total), **f64), torch.zeros((HKV, total), **f64)
    lost, error = torch.zeros((case.get("specs", 1), total), **f64), torch.zeros(count, **f64)
    counters = torch.zeros(total, **f64)
    seen = None
    if kind == "replay" and start > case["budget"]:
        seen = torch.zeros((HKV, total), dtype=torch.bool, device="cuda")
        seen[:, start:] = True
        seen.scatter_(1, x.kept, True)
    for first in range(0, count, step):
        at_q = torch.arange(first, min(count, first + step), device="cuda")
        hidden = place > at_q[:, None] + start
        credit = torch.zeros((len(at_q), total), **f64)
        diff = same = 0.0
        for g in range(HKV):
            q = x.q[at_q, g * GROUP:(g + 1) * GROUP].double().transpose(0, 1)  # [j, q, d]
            logits = (torch.matmul(q, keys[:, g].t().contiguous()) * SCALE).masked_fill(hidden, float("-inf"))
            sink = x.sinks[g * GROUP:(g + 1) * GROUP].double()[:, None, None]

            def probability(z):
                return torch.exp(z - torch.logaddexp(torch.logsumexp(z, -1, keepdim=True), sink))
            p = probability(logits)
            if kind == "replay":
                if seen is not None:
                    a = torch.matmul(p, values[:, g])
                    b = torch.matmul(probability(logits.masked_fill(~seen[g], float("-inf"))), values[:, g])
                    diff, same = diff + (b - a).square().sum((0, 2)), same + a.square().sum((0, 2))
                continue
            sums[g] += p.sum((0, 1))
            maxes[g] += p.amax(0).sum(0)
            credit = torch.maximum(credit, p.amax(0))
            if kind == "diagnose":
                for j in range(case["specs"]):
                    gone = ~x.resident[j, 0, g]
                    lost[j, start + at_q] += p[..., gone].sum((0, 2)) / HQ
        if kind == "replay" and seen is not None:
            error[at_q] = diff.sqrt() / same.sqrt().clamp_min(1e-12)
        if kind == "counters":
            block = case["block"]
            whole = (at_q + start + 1 - case["delay"]).clamp_min(0) // block  # blocks a query credits
            n = total // block
            best = credit[:, :n * block].view(len(at_q), n, block).amax(-1)
            best = best * (torch.arange(n, device="cuda") < whole[:, None])
            counters[:n * block:block] += best.sum(0)
    if kind == "replay":
        return {"error": error}
    if kind == "diagnose":
        return {"score_sum": sums[None], "score_max": maxes[None], "lost": lost}
    scores = torch.zeros((1, HKV, x.size), **f64)
    if kind == "counters":
        scores[0, 0, at] = counters
    else:
        scores[0, :, at] = sums if case["policy"] == "head_sum_2048" else maxes
    return {"scores": scores}
