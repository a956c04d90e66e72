"""Decode path on the GPU through the C ABI: CSR fill, fused attention + scores, and the
reference hook `after_decode`, against the CPU oracle."""
from types import SimpleNamespace

import numpy as np
import pytest
import torch

import oracle as O
from fakes import backend, layer

pytestmark = pytest.mark.gpu

ge = None


@pytest.fixture(autouse=True)
def fresh_state():
    global ge
    if not torch.cuda.is_available():
        pytest.skip("needs a GPU")
    import gstar_evict
    ge = gstar_evict
    ge.STATE = None
    yield
    ge.STATE = None


# T:80-90's known answer: row 1 holds 4 compacted slots below frontier 7 and reads req_to_token
# from 7 up to its length 10; row 2 (length 6) has had no boundary.
FILL_KNOWN = dict(r2t={1: list(range(101, 111)), 2: list(range(201, 207))}, table={1: [101, 102, 106, 107]},
                  count={1: 4}, frontier={1: 7}, rows=[1, 2], lens=[10, 6], indptr=[0, 7, 13],
                  indices=[101, 102, 106, 107, 108, 109, 110, 201, 202, 203, 204, 205, 206])


def test_fill_reads_compact_residents_then_tail():
    b = backend()
    st = ge.state(b)
    case = FILL_KNOWN
    for row, slots in case["r2t"].items():
        st.req_to_token[row, :len(slots)] = torch.tensor(slots, dtype=torch.int32)
    for row, slots in case["table"].items():
        st.table[row, :len(slots)] = torch.tensor(slots, dtype=torch.int32)
        st.count[row], st.frontier[row] = case["count"][row], case["frontier"][row]
    for dtype in (torch.int64, torch.int32):  # index tensors of either width
        out = torch.full((32,), -1, dtype=dtype, device="cuda")
        as_dev = lambda v: torch.tensor(v, dtype=dtype, device="cuda")
        indptr = ge.fill(b, 2, as_dev(case["lens"]), as_dev(case["rows"]), out)
        assert indptr.tolist() == case["indptr"]
        assert out[:len(case["indices"])].tolist() == case["indices"]


def test_fill_matches_oracle_on_random_rows():
    g = torch.Generator().manual_seed(11)
    b = backend(rows=8, width=4096)
    st = ge.state(b)
    st.req_to_token.copy_(torch.randint(1, 20000, (8, 4096), generator=g, dtype=torch.int32))
    st.table.copy_(torch.randint(1, 20000, (8, 4096), generator=g, dtype=torch.int32))
    count = torch.randint(0, 1000, (8,), generator=g, dtype=torch.int32)
    frontier = count + torch.randint(0, 500, (8,), generator=g, dtype=torch.int32)
    st.count.copy_(count)
    st.frontier.copy_(frontier)
    rows = torch.tensor([5, 0, 7, 2, 3], device="cuda")
    lens = frontier[rows.cpu()].long() + torch.randint(0, 2000, (5,), generator=g)
    out = torch.full((40000,), -1, dtype=torch.int32, device="cuda")
    indptr = ge.fill(b, 5, lens.cuda(), rows, out)
    want_ptr, want = O.fill(st.table.cpu().numpy(), st.req_to_token.cpu().numpy(), rows.cpu().numpy(),
                            lens.numpy(), frontier.numpy(), count.numpy())
    assert indptr.tolist() == want_ptr.tolist()
    assert out[:want.size].tolist() == want.tolist()


def _decode_setup(lengths, seed=0, slots=20000):
    g = torch.Generator().manual_seed(seed)
    b = backend(gen=g, slots=slots, rows=max(4, len(lengths) + 1))  # rows 1..bs
    st = ge.state(b)
    heads, kv_heads, dim = 64, 8, 64
    bs = len(lengths)
    q = torch.randn((bs, heads, dim), generator=g).to(torch.bfloat16).cuda()
    sinks = torch.randn(heads, generator=g).to(torch.bfloat16).cuda()
    assert sum(lengths) < slots
    perm = (torch.randperm(slots - 1, generator=g)[:sum(lengths)] + 1).cuda()
    indptr = torch.tensor(np.concatenate(([0], np.cumsum(lengths))), dtype=torch.int32, device="cuda")
    rows = torch.arange(1, bs + 1, device="cuda")
    return b, st, q, sinks, perm, indptr, rows


def _oracle_step(b, st, q, sinks, perm, indptr, lid, mode, delay=0):
    """Each sequence's attention and scores; its list holds positions 0..len-1 (no boundary yet),
    so a score delay credits the keys at least `delay` positions before the query (len - 1)."""
    keys = b.token_to_kv_pool.get_key_buffer(lid).float().cpu().numpy()
    values = b.token_to_kv_pool.get_value_buffer(lid).float().cpu().numpy()
    qn = q.float().cpu().numpy()
    s = sinks.float().cpu().numpy()
    ip = indptr.cpu().numpy()
    pm = perm.cpu().numpy()
    outs, norms = [], []
    scores = np.zeros((st.kv_heads, keys.shape[0]))
    for i in range(q.shape[0]):
        slots = pm[ip[i]:ip[i + 1]]
        o, norm = O.decode_attention(qn[i], keys, values, slots, s, 0.125)
        outs.append(o)
        norms.append(norm)
        O.decode_scores_into(scores, qn[i], keys, slots, norm, 0.125, mode, np.arange(len(slots)), len(slots) - 1,
                             delay)
    return np.stack(outs), np.stack(norms), scores


@pytest.mark.parametrize("mode", [1, 2])
@pytest.mark.parametrize("queued", [False, True])
@pytest.mark.parametrize("delay", [0, 100])
def test_fused_decode_matches_oracle(mode, queued, delay):
    """Attention and scores; a score delay of 100 (block policies) leaves the 37-key list unscored
    and the others' newest 100 keys."""
    lengths = [37, 1500, 3001]
    b, st, q, sinks, perm, indptr, rows = _decode_setup(lengths)
    st.score_mode = "queue" if queued else "eager"
    st.mode[:] = mode | delay << 8
    b.forward_metadata = SimpleNamespace(kv_indptr=indptr, kv_indices=perm)
    fb = SimpleNamespace(out_cache_loc=torch.zeros(3, dtype=torch.int64, device="cuda"), req_pool_indices=rows,
                         seq_lens_cpu=torch.tensor(lengths))
    o = torch.empty_like(q)
    assert ge.decode(b, q.reshape(3, -1), layer(1), fb, sinks, o.reshape(3, -1))
    if queued:
        assert float(st.scores.abs().sum()) == 0.0  # the step is queued until flushed
        # The flush rebuilds each row's list from the eviction state (empty table, tail = req_to_token).
        for i, r in enumerate(rows.tolist()):
            st.req_to_token[r, :lengths[i]] = perm[indptr[i]:indptr[i + 1]].int()
        ge.flush(st)
    want_o, want_norm, want_scores = _oracle_step(b, st, q, sinks, perm, indptr, 1, mode, delay)
    got_o = o.float().cpu().numpy()
    # bf16 output: P is rounded to bf16 before the PV product, as in SGLang's decode kernel.
    np.testing.assert_allclose(got_o, want_o, rtol=2e-2, atol=2e-2)
    assert np.abs(got_o - want_o).mean() < 2e-3
    expected = torch.zeros_like(st.scores)
    expected[0] = torch.tensor(want_scores, dtype=torch.float32)
    torch.testing.assert_close(st.scores, expected, rtol=2e-3, atol=1e-6)


def test_queue_over_steps_equals_eager():
    """Several decode steps with growing lists: queued + flushed scores equal eager ones."""
    g = torch.Generator().manual_seed(3)
    results = {}
    for queued in (False, True):
        ge.STATE = None
        b = backend(gen=torch.Generator().manual_seed(1))
        st = ge.state(b)
        st.score_mode = "queue" if queued else "eager"
        st.mode[:] = 1
        base = [100, 700]
        perm = (torch.randperm(19999, generator=torch.Generator().manual_seed(2))[:2000] + 1).cuda()
        qs = [torch.randn((2, 64, 64), generator=torch.Generator().manual_seed(10 + t)).to(torch.bfloat16).cuda()
              for t in range(4)]
        sinks = torch.randn(64, generator=torch.Generator().manual_seed(5)).cuda()
        for t in range(4):
            lens = [base[0] + t, base[1] + t]
            idx = torch.cat((perm[:lens[0]], perm[1000:1000 + lens[1]]))
            indptr = torch.tensor([0, lens[0], lens[0] + lens[1]], dtype=torch.int32, device="cuda")
            b.forward_metadata = SimpleNamespace(kv_indptr=indptr, kv_indices=idx)
            fb = SimpleNamespace(out_cache_loc=idx[indptr[1:].long() - 1], req_pool_indices=torch.tensor(
                [1, 2], device="cuda"), seq_lens_cpu=torch.tensor(lens))
            o = torch.empty((2, 64, 64), dtype=torch.bfloat16, device="cuda")
            ge.decode(b, qs[t].reshape(2, -1), layer(1), fb, sinks, o.reshape(2, -1))
        # Flushing needs the row view of the lists: table empty, tail = req_to_token.
        st.req_to_token[1, :base[0] + 3] = perm[:base[0] + 3].int()
        st.req_to_token[2, :base[1] + 3] = perm[1000:1000 + base[1] + 3].int()
        ge.flush(st)
        results[queued] = st.scores.clone()
    # Only the fp32 summation order differs (per step vs per queue).
    torch.testing.assert_close(results[True], results[False], rtol=1e-5, atol=1e-8)


def _fold_case(name):
    """(lengths, score words, folded batch indices) of a fold case: four sequences (the merge's
    8-group instance), two long ones (64 groups per head: a third of P or more per sequence) and
    40 short ones (one group per head)."""
    if name == "bs4":
        return [2000, 37, 5000, 900], [1, 2, 1 | 64 << 8, 1], [0, 1, 2]
    if name == "bs2":
        return [5000, 4500], [2 | 64 << 8, 1], [0]
    g = np.random.default_rng(40)
    lengths = [int(x) for x in g.integers(30, 400, size=40)]
    modes = [2 if i % 5 == 3 else 1 for i in range(40)]
    return lengths, modes, [0, 7, 13]


@pytest.mark.parametrize("case,queued", [("bs4", 1), ("bs4", 20), ("bs4", 63), ("bs2", 20), ("bs40", 5)])
def test_in_launch_fold_equals_the_long_flush(case, queued):
    """A decode launch's fold workgroups add a queue exactly as gse_score_flush does (the same
    tiles, chunks and atomics: bit for bit), for sum and max rows and a score delay, and the
    launch's own step restarts each folded queue (entry 0, count 1); an unlisted row keeps its
    queue. The merge that scatters the fold's totals runs each of its instances: four sequences
    (8 groups of 8 heads), two sequences of about 5K keys over some 157 workgroups (64 groups
    per head), and 40 short sequences (one group per head)."""
    lengths0, modes, folded = _fold_case(case)
    bs = len(lengths0)
    b = backend(gen=torch.Generator().manual_seed(11), rows=bs + 2)
    st = ge.state(b)
    st.score_mode = "queue"
    rows = torch.arange(1, bs + 1, device="cuda")
    for i, m in enumerate(modes):
        st.entries[i + 1] = {"mode": m & 0xff}
        st.mode[i + 1] = m
    g = torch.Generator().manual_seed(12)
    total = sum(lengths0) + bs * (queued + 1)
    assert total < 19999
    perm = (torch.randperm(19999, generator=g)[:total] + 1).cuda()
    offs = np.concatenate(([0], np.cumsum([n + queued + 1 for n in lengths0])))
    for i, n in enumerate(lengths0):
        st.req_to_token[i + 1, :n + queued + 1] = perm[offs[i]:offs[i + 1]].int()
    sinks = torch.randn(64, generator=g).cuda()
    qs = [torch.randn((bs, 64, 64), generator=g).to(torch.bfloat16).cuda() for _ in range(queued + 1)]

    def step(t):
        lens = [n + t + 1 for n in lengths0]
        idx = torch.cat([perm[offs[i]:offs[i] + lens[i]] for i in range(bs)])
        indptr = torch.tensor(np.concatenate(([0], np.cumsum(lens))), dtype=torch.int32, device="cuda")
        b.forward_metadata = SimpleNamespace(kv_indptr=indptr, kv_indices=idx)
        fb = SimpleNamespace(out_cache_loc=torch.zeros(bs, dtype=torch.int64, device="cuda"), req_pool_indices=rows,
                             seq_lens_cpu=torch.tensor(lens))
        o = torch.empty((bs, 64, 64), dtype=torch.bfloat16, device="cuda")
        ge.decode(b, qs[t].reshape(bs, -1), layer(1), fb, sinks, o.reshape(bs, -1))

    for t in range(queued):
        step(t)
    torch.cuda.synchronize()
    assert st.qcount[0, 1:bs + 1].tolist() == [queued] * bs
    saved = [x.clone() for x in (st.scores, st.qq, st.qnorm, st.qlim, st.qcount)]
    st.queued = {r: queued for r in range(1, bs + 1)}
    ge.flush(st, [i + 1 for i in folded])
    flushed = st.scores.clone()
    assert float((flushed - saved[0]).abs().sum()) > 0
    for dst, src in zip((st.scores, st.qq, st.qnorm, st.qlim, st.qcount), saved):
        dst.copy_(src)
    st.fold_seq, st.fold_n = st.fold_list(folded), len(folded)
    step(queued)
    torch.cuda.synchronize()
    assert torch.equal(st.scores, flushed)
    assert st.qcount[0, 1:bs + 1].tolist() == [1 if i in folded else queued + 1 for i in range(bs)]
    for i in range(bs):
        entry = 0 if i in folded else queued
        assert torch.equal(st.qq[0, i + 1, entry], qs[queued][i])
        assert int(st.qlim[0, i + 1, entry]) == lengths0[i] + queued + 1


@pytest.mark.parametrize("steps,delay,kv_heads", [(1, 0, 8), (5, 0, 8), (8, 64, 8), (13, 0, 8), (3, 7, 4)])
def test_short_and_long_queue_flushes_agree(monkeypatch, steps, delay, kv_heads):
    """The short-queue flush (a workgroup reads every KV head of its keys, one score-row write
    per slot) and the long-queue flush fold the same queued steps (rows of sum and max mode,
    growing lists) to the same scores, and both equal the eager per-step update. 13 steps take
    the short kernel's restaging path; 4 KV heads its per-head score writes."""
    from gstar_evict import attention
    heads = 8 * kv_heads
    results = {}
    for which in ("long", "short", "eager"):
        monkeypatch.setattr(attention, "SHORT_QUEUE", 64 if which == "short" else -1)
        ge.STATE = None
        b = backend(gen=torch.Generator().manual_seed(1), kv_heads=kv_heads)
        st = ge.state(b)
        st.score_mode = "eager" if which == "eager" else "queue"
        st.mode[1], st.mode[2] = 1 | delay << 8, 2 | delay << 8
        base = [100, 1301]
        perm = (torch.randperm(19999, generator=torch.Generator().manual_seed(2))[:3000] + 1).cuda()
        sinks = torch.randn(heads, generator=torch.Generator().manual_seed(5)).cuda()
        for t in range(steps):
            q = torch.randn((2, heads, 64), generator=torch.Generator().manual_seed(10 + t)).to(torch.bfloat16).cuda()
            lens = [base[0] + t, base[1] + t]
            idx = torch.cat((perm[:lens[0]], perm[1500:1500 + lens[1]]))
            indptr = torch.tensor([0, lens[0], lens[0] + lens[1]], dtype=torch.int32, device="cuda")
            b.forward_metadata = SimpleNamespace(kv_indptr=indptr, kv_indices=idx)
            fb = SimpleNamespace(out_cache_loc=idx[indptr[1:].long() - 1], req_pool_indices=torch.tensor(
                [1, 2], device="cuda"), seq_lens_cpu=torch.tensor(lens))
            o = torch.empty((2, heads, 64), dtype=torch.bfloat16, device="cuda")
            lay = layer(1, heads=heads, kv_heads=kv_heads)
            ge.decode(b, q.reshape(2, -1), lay, fb, sinks, o.reshape(2, -1))
        st.req_to_token[1, :base[0] + steps] = perm[:base[0] + steps].int()
        st.req_to_token[2, :base[1] + steps] = perm[1500:1500 + base[1] + steps].int()
        ge.flush(st)
        results[which] = st.scores.clone()
    assert float(results["long"].abs().sum()) > 0
    torch.testing.assert_close(results["short"], results["long"], rtol=1e-6, atol=1e-9)
    torch.testing.assert_close(results["short"], results["eager"], rtol=1e-5, atol=1e-8)


@pytest.mark.parametrize("mode,delay", [(1, 0), (2, 0), (1, 64)])
def test_after_decode_rebuilds_normaliser_from_split_lse(mode, delay):
    """T:48-78 with SGLang's split LSE layout (splits [1, 5, 8]) produced by the oracle; with a
    score delay the newest `delay` keys of each list get nothing."""
    lengths = [37, 1500, 3001]
    b, st, q, sinks, perm, indptr, rows = _decode_setup(lengths, seed=4)
    splits = [1, 5, 8]
    keys = b.token_to_kv_pool.get_key_buffer(1).float().cpu().numpy()
    lse = np.zeros((3, 64, 8), dtype=np.float32)
    for i in range(3):
        logits = O.decode_logits(q[i].float().cpu().numpy(), keys, perm[indptr[i]:indptr[i + 1]].cpu().numpy(), 0.125)
        part, _ = O.split_lse(logits, splits[i])
        lse[i, :, :splits[i]] = np.nan_to_num(part, nan=1e30)
    b.forward_metadata = SimpleNamespace(attn_lse=torch.tensor(lse, device="cuda"), kv_indptr=indptr,
                                         kv_indices=perm, num_kv_splits=torch.tensor(splits, dtype=torch.int32,
                                                                                      device="cuda"))
    st.mode[:] = mode | delay << 8
    ge.after_decode(b, q.reshape(3, -1), layer(1), SimpleNamespace(
        out_cache_loc=torch.zeros(3, dtype=torch.int64, device="cuda"), req_pool_indices=rows), sinks)
    expected = np.zeros(tuple(st.scores.shape[1:]))
    for i in range(3):
        rows_keys = perm[indptr[i]:indptr[i + 1]].cpu().numpy()
        qn = q[i].float().cpu().numpy()
        _, norm = O.decode_attention(qn, keys, keys, rows_keys, sinks.float().cpu().numpy(), 0.125)
        O.decode_scores_into(expected, qn, keys, rows_keys, norm, 0.125, mode, np.arange(len(rows_keys)),
                             len(rows_keys) - 1, delay)
    torch.testing.assert_close(st.scores[0].cpu(), torch.tensor(expected, dtype=torch.float32), rtol=2e-3, atol=1e-6)
    assert float(st.scores[1:].abs().sum()) == 0.0


# The pass cuts all lists into one range of 64-key tiles: lists that are empty, end on a tile's edge
# or one past it, more than the 64 lists of one scan, unscored rows between, and split counts past
# the 16 the first loads cover.
@pytest.mark.parametrize("lengths,splits", [([1], 1), ([64], 2), ([65, 0, 63], 8), ([0, 0, 5000, 0, 1], 17),
                                            ([130, 64, 0, 1, 65, 300] * 23 + [129], 40)])
def test_after_decode_over_many_lists(lengths, splits):
    bs = len(lengths)
    b, st, q, sinks, perm, indptr, rows = _decode_setup(lengths, seed=bs + splits)
    b.max_kv_splits = splits
    kinds = [1, 2, 0]
    st.mode[:] = 0
    st.mode[rows.long()] = torch.tensor([kinds[i % 3] for i in range(bs)], dtype=torch.int32, device="cuda")
    keys = b.token_to_kv_pool.get_key_buffer(1)
    lse = torch.full((bs, 64, splits), 1e30, device="cuda")  # splits past a list's end are never read
    want = torch.zeros(tuple(st.scores.shape[1:]), dtype=torch.float64, device="cuda")
    for i, n in enumerate(lengths):
        if not n:
            continue
        slots = perm[indptr[i]:indptr[i + 1]].long()
        per = -(-(-(-n // splits)) // 32) * 32
        x = torch.matmul(q[i].double().view(8, 8, 64), keys[slots].double().permute(1, 2, 0).contiguous()) * 0.125
        for s in range(-(-n // per)):
            lse[i, :, s] = torch.logsumexp(x[..., s * per:(s + 1) * per], -1).reshape(64).float()
        norm = torch.logaddexp(torch.logsumexp(x, -1), sinks.double().view(8, 8))
        p = torch.exp(x - norm[..., None])
        if kinds[i % 3]:
            want[:, slots] += p.sum(1) if kinds[i % 3] == 1 else p.amax(1)
    b.forward_metadata = SimpleNamespace(attn_lse=lse, kv_indptr=indptr, kv_indices=perm, num_kv_splits=torch.full(
        (bs,), splits, dtype=torch.int32, device="cuda"))
    ge.after_decode(b, q.reshape(bs, -1), layer(1), SimpleNamespace(
        out_cache_loc=torch.zeros(bs, dtype=torch.int64, device="cuda"), req_pool_indices=rows,
        seq_lens_cpu=torch.tensor(lengths)), sinks)
    # 32-bit logits and log-sum-exps of magnitude up to about 16: 2^-20 each.
    torch.testing.assert_close(st.scores[0].double(), want, rtol=1e-5, atol=1e-8)


def test_rows_without_a_policy_get_no_scores_and_sliding_layers_are_skipped():
    lengths = [64, 65]
    b, st, q, sinks, perm, indptr, rows = _decode_setup(lengths, seed=6)
    st.mode[:] = 0
    st.mode[2] = 2
    st.score_mode = "eager"
    b.forward_metadata = SimpleNamespace(kv_indptr=indptr, kv_indices=perm)
    fb = SimpleNamespace(out_cache_loc=torch.zeros(2, dtype=torch.int64, device="cuda"), req_pool_indices=rows,
                         seq_lens_cpu=torch.tensor(lengths))
    o = torch.empty_like(q)
    assert not ge.decode(b, q.reshape(2, -1), SimpleNamespace(**{**vars(layer(0)), "sliding_window_size": 128}),
                         fb, sinks, o.reshape(2, -1))
    ge.decode(b, q.reshape(2, -1), layer(3), fb, sinks, o.reshape(2, -1))
    touched = st.scores[1].abs().sum(0) > 0
    assert not bool(touched[perm[:64]].any())
    assert bool(touched[perm[64:]].all())
    assert float(st.scores[0].abs().sum()) == 0.0


@pytest.mark.parametrize("mode", [1, 2])
def test_full_queues_flush_before_the_step(monkeypatch, mode):
    """More steps than the queue holds: begin_decode_step flushes full queues, so queued +
    flushed scores equal the eager per-step update (head-sum and head-max)."""
    monkeypatch.setenv("GSTAR_EVICT_QUEUE", "3")
    results = {}
    steps, base = 8, [130, 900]
    perm = (torch.randperm(19999, generator=torch.Generator().manual_seed(12))[:2000] + 1).cuda()
    qs = [torch.randn((2, 64, 64), generator=torch.Generator().manual_seed(40 + t)).to(torch.bfloat16).cuda()
          for t in range(steps)]
    sinks = torch.randn(64, generator=torch.Generator().manual_seed(7)).cuda()
    for score_mode in ("eager", "queue"):
        ge.STATE = None
        b = backend(gen=torch.Generator().manual_seed(9))
        st = ge.state(b)
        assert st.queue_cap == 3
        st.score_mode = score_mode
        for r in (1, 2):
            st.entries[r] = {"mode": mode}
            st.mode[r] = mode
        st.req_to_token[1, :base[0] + steps] = perm[:base[0] + steps].int()
        st.req_to_token[2, :base[1] + steps] = perm[1000:1000 + base[1] + steps].int()
        for t in range(steps):
            lens = [base[0] + t, base[1] + t]
            idx = torch.cat((perm[:lens[0]], perm[1000:1000 + lens[1]]))
            indptr = torch.tensor([0, lens[0], lens[0] + lens[1]], dtype=torch.int32, device="cuda")
            b.forward_metadata = SimpleNamespace(kv_indptr=indptr, kv_indices=idx)
            fb = SimpleNamespace(out_cache_loc=idx[indptr[1:].long() - 1], req_pool_indices=torch.tensor(
                [1, 2], device="cuda"), seq_lens_cpu=torch.tensor(lens))
            ge.begin_decode_step([1, 2], st)
            if score_mode == "queue":
                assert max(st.queued.values()) <= st.queue_cap
            o = torch.empty((2, 64, 64), dtype=torch.bfloat16, device="cuda")
            ge.decode(b, qs[t].reshape(2, -1), layer(1), fb, sinks, o.reshape(2, -1))
        assert int(st.qcount.max()) <= st.queue_cap  # no step was dropped
        ge.flush(st)
        assert int(st.qcount.abs().sum()) == 0
        results[score_mode] = st.scores.clone()
    torch.testing.assert_close(results["queue"], results["eager"], rtol=1e-5, atol=1e-8)


def test_merge_of_empty_short_and_long_sequences_over_a_reused_workspace():
    """The merge of a batch with empty sequences (all mass on the sink: o = 0, normaliser =
    sink, queued with list length 0), one inside a single workgroup and one across many; then a
    smaller batch on the same workspace. Each row's queue count is exactly one step."""
    for call, lengths in enumerate(([0, 5, 4000, 0, 1], [300, 2])):
        b, st, q, sinks, perm, indptr, rows = _decode_setup(lengths, seed=20 + call)
        if call:
            st._ws = keep  # the previous call's workspace
        st.score_mode = "queue"
        st.mode[:] = 1
        b.forward_metadata = SimpleNamespace(kv_indptr=indptr, kv_indices=perm)
        fb = SimpleNamespace(out_cache_loc=torch.zeros(len(lengths), dtype=torch.int64, device="cuda"),
                             req_pool_indices=rows, seq_lens_cpu=torch.tensor(lengths))
        o = torch.full_like(q, float("nan"))
        assert ge.decode(b, q.reshape(len(lengths), -1), layer(1), fb, sinks, o.reshape(len(lengths), -1))
        keep = st._ws
        got = o.float().cpu().numpy()
        keys = b.token_to_kv_pool.get_key_buffer(1).float().cpu().numpy()
        values = b.token_to_kv_pool.get_value_buffer(1).float().cpu().numpy()
        ip, pm, sn = indptr.cpu().numpy(), perm.cpu().numpy(), sinks.float().cpu().numpy()
        index = st.index[1]
        for i, n in enumerate(lengths):
            row = int(rows[i])
            assert int(st.qcount[index, row]) == 1
            assert int(st.qlim[index, row, 0]) == n
            if n == 0:
                assert np.all(got[i] == 0.0)
                np.testing.assert_allclose(st.qnorm[index, row, 0].cpu().numpy(), sn, rtol=1e-6, atol=1e-6)
                continue
            want_o, want_norm = O.decode_attention(q[i].float().cpu().numpy(), keys, values, pm[ip[i]:ip[i + 1]], sn,
                                                   0.125)
            np.testing.assert_allclose(got[i], want_o, rtol=2e-2, atol=2e-2)
            np.testing.assert_allclose(st.qnorm[index, row, 0].cpu().numpy(), want_norm, rtol=1e-5, atol=1e-4)
        assert torch.equal(st.qq[index, rows, 0], q)
        ge.STATE = None


# Batches whose workgroups each keep to one sequence (2 to 32 sequences, at least 8 workgroups per
# sequence), at the edges of that rule and of the shares: empty lists, one key, all of the keys in one
# list; then more sequences than workgroups (one tile in all), where a workgroup counts several rows.
@pytest.mark.parametrize("lengths", [
    [1, 1], [0, 5000], [6000, 0], [700] * 3 + [1], [2047, 2049, 0, 64, 63], [513] * 8, [300] * 31 + [0],
    [600] * 32, [600] * 33, [1] * 40, [0] * 20 + [3] + [0] * 20])
def test_workgroups_of_one_sequence_each(lengths):
    bs = len(lengths)
    b, st, q, sinks, perm, indptr, rows = _decode_setup(lengths, seed=bs + sum(lengths), slots=24000)
    st.score_mode = "queue"
    kinds = torch.tensor([i % 3 for i in range(bs)], dtype=torch.int32, device="cuda")  # kind 0: not queued
    st.mode[:] = 0
    st.mode[rows] = kinds
    b.forward_metadata = SimpleNamespace(kv_indptr=indptr, kv_indices=perm)
    fb = SimpleNamespace(out_cache_loc=torch.zeros(bs, dtype=torch.int64, device="cuda"), req_pool_indices=rows,
                         seq_lens_cpu=torch.tensor(lengths))
    o = torch.full_like(q, float("nan"))
    for step in range(2):
        assert ge.decode(b, q.reshape(bs, -1), layer(1), fb, sinks, o.reshape(bs, -1))
    index = st.index[1]
    keys, values = (f(1) for f in (b.token_to_kv_pool.get_key_buffer, b.token_to_kv_pool.get_value_buffer))
    counts = torch.where(kinds > 0, 2, 0).to(torch.int32)
    assert torch.equal(st.qcount[index, rows], counts)
    assert int(st.qcount[index].sum()) == int(counts.sum())  # no other row's moved
    for i, n in enumerate(lengths):
        slots = perm[indptr[i]:indptr[i + 1]].long()
        x = torch.matmul(q[i].double().view(8, 8, 64), keys[slots].double().permute(1, 2, 0).contiguous()) * 0.125
        sink = sinks.double().view(8, 8)
        norm = torch.logaddexp(torch.logsumexp(x, -1), sink) if n else sink
        want = torch.matmul(torch.exp(x - norm[..., None]), values[slots].double().transpose(0, 1).contiguous())
        # Probabilities and outputs are rounded to bf16 (2^-9 each); values are N(0, 1).
        torch.testing.assert_close(o[i].double(), want.reshape(64, 64), rtol=8e-3, atol=8e-3)
        if kinds[i]:
            for entry in range(2):
                torch.testing.assert_close(st.qnorm[index, rows[i], entry].double(), norm.reshape(64), rtol=1e-6,
                                           atol=4e-6)
                assert int(st.qlim[index, rows[i], entry]) == n
                assert torch.equal(st.qq[index, rows[i], entry], q[i])


# A workgroup's chunk never takes more 64-key tile steps than an even cut of the batch over the same
# grid would: lists whose shares fit in whole tiles, and a batch whose shares would not (its last
# tiles exceed the chip's workgroups) and is cut evenly.
@pytest.mark.parametrize("lengths", [[4000] * 2, [4000] * 4, [8000, 7980], [16084, 100, 100, 100], [0, 8192, 0, 8191]])
def test_shares_by_sequence_take_no_more_tile_steps_than_an_even_cut(lengths):
    bs, total = len(lengths), sum(lengths)
    b, st, q, sinks, perm, indptr, rows = _decode_setup(lengths, seed=total)
    b.forward_metadata = SimpleNamespace(kv_indptr=indptr, kv_indices=perm)
    fb = SimpleNamespace(out_cache_loc=torch.zeros(bs, dtype=torch.int64, device="cuda"), req_pool_indices=rows,
                         seq_lens_cpu=torch.tensor(lengths))
    o = torch.empty_like(q)
    ge.decode(b, q.reshape(bs, -1), layer(1), fb, sinks, o.reshape(bs, -1))  # the workspace is there
    ws = st._ws["decode"]
    ws.fill_(255)  # NaN partials
    ge.decode(b, q.reshape(bs, -1), layer(1), fb, sinks, o.reshape(bs, -1))
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    grid = min(cus, -(-bs * max(lengths) // 64))
    steps = -(-(-(-total // grid)) // 64)
    partials = ws[:(cus + bs) * 64 * 68 * 4].view(torch.float32).view(-1, 64, 68)  # o[64], m, l, pad per head
    used = int((~partials[:, 0, 64].isnan()).sum())
    assert used * 64 * steps >= total
    keys, values = (f(1) for f in (b.token_to_kv_pool.get_key_buffer, b.token_to_kv_pool.get_value_buffer))
    for i, n in enumerate(lengths):
        slots = perm[indptr[i]:indptr[i + 1]].long()
        x = torch.matmul(q[i].double().view(8, 8, 64), keys[slots].double().permute(1, 2, 0).contiguous()) * 0.125
        sink = sinks.double().view(8, 8)
        norm = torch.logaddexp(torch.logsumexp(x, -1), sink) if n else sink
        want = torch.matmul(torch.exp(x - norm[..., None]), values[slots].double().transpose(0, 1).contiguous())
        # As above: bf16 probabilities and outputs.
        torch.testing.assert_close(o[i].double(), want.reshape(64, 64), rtol=8e-3, atol=8e-3)


@pytest.mark.parametrize("bs", [40, 5, 3, 1, 300])
def test_merge_paths_for_many_and_few_sequences(bs):
    """The merge folds a sequence's partials in one group when there are at least 32 sequences
    (about 8 workgroups each), in 8 groups of 8 heads combined through LDS down to 4 sequences,
    and below that (one to three sequences, each spread over up to 256 workgroups) in 64 groups
    per head, folded in two levels: all against the oracle, outputs and queued normalisers (the
    queue count advanced once by 64 head workgroups). With more sequences than workgroups (300
    lists of 0-59 keys), a workgroup's range holds several whole sequences, empty ones included."""
    g = np.random.default_rng(bs)
    lo, hi = (0, 60) if bs > 256 else (1, 400 if bs > 8 else 6000)
    lengths = [int(x) for x in g.integers(lo, hi, size=bs)]
    b, st, q, sinks, perm, indptr, rows = _decode_setup(lengths, seed=30 + bs, slots=40000)
    st.score_mode = "queue"
    st.mode[:] = 1
    b.forward_metadata = SimpleNamespace(kv_indptr=indptr, kv_indices=perm)
    fb = SimpleNamespace(out_cache_loc=torch.zeros(bs, dtype=torch.int64, device="cuda"), req_pool_indices=rows,
                         seq_lens_cpu=torch.tensor(lengths))
    o = torch.empty_like(q)
    assert ge.decode(b, q.reshape(bs, -1), layer(1), fb, sinks, o.reshape(bs, -1))
    keys = b.token_to_kv_pool.get_key_buffer(1).float().cpu().numpy()
    values = b.token_to_kv_pool.get_value_buffer(1).float().cpu().numpy()
    ip, pm, sn = indptr.cpu().numpy(), perm.cpu().numpy(), sinks.float().cpu().numpy()
    got = o.float().cpu().numpy()
    index = st.index[1]
    norms = st.qnorm[index, 1:bs + 1, 0].cpu().numpy()
    for i in range(bs):
        if lengths[i] == 0:  # all mass on the sink
            assert np.all(got[i] == 0.0)
            np.testing.assert_allclose(norms[i], sn, rtol=1e-6, atol=1e-6)
            continue
        want_o, want_norm = O.decode_attention(q[i].float().cpu().numpy(), keys, values, pm[ip[i]:ip[i + 1]], sn, 0.125)
        np.testing.assert_allclose(got[i], want_o, rtol=2e-2, atol=2e-2)
        np.testing.assert_allclose(norms[i], want_norm, rtol=1e-5, atol=1e-4)
    assert st.qcount[index, 1:bs + 1].tolist() == [1] * bs


@pytest.mark.parametrize("length", [1, 37, 64, 65, 129])
def test_single_short_sequence_on_one_to_three_workgroups(length):
    """A bs=1 call of n keys runs on ceil(n / 64) attention workgroups (one 64-key tile each):
    1, 37 and 64 keys on one, 65 on two, 129 on three; outputs, the queued normaliser and the
    queued step against the oracle."""
    b, st, q, sinks, perm, indptr, rows = _decode_setup([length], seed=50 + length)
    st.score_mode = "queue"
    st.mode[:] = 1
    b.forward_metadata = SimpleNamespace(kv_indptr=indptr, kv_indices=perm)
    fb = SimpleNamespace(out_cache_loc=torch.zeros(1, dtype=torch.int64, device="cuda"), req_pool_indices=rows,
                         seq_lens_cpu=torch.tensor([length]))
    o = torch.full_like(q, float("nan"))
    assert ge.decode(b, q.reshape(1, -1), layer(1), fb, sinks, o.reshape(1, -1))
    keys = b.token_to_kv_pool.get_key_buffer(1).float().cpu().numpy()
    values = b.token_to_kv_pool.get_value_buffer(1).float().cpu().numpy()
    want_o, want_norm = O.decode_attention(q[0].float().cpu().numpy(), keys, values, perm.cpu().numpy(),
                                           sinks.float().cpu().numpy(), 0.125)
    index = st.index[1]
    np.testing.assert_allclose(o[0].float().cpu().numpy(), want_o, rtol=2e-2, atol=2e-2)
    np.testing.assert_allclose(st.qnorm[index, 1, 0].cpu().numpy(), want_norm, rtol=1e-5, atol=1e-4)
    assert int(st.qcount[index, 1]) == 1 and int(st.qlim[index, 1, 0]) == length
    assert torch.equal(st.qq[index, 1, 0], q[0])
