"""Chunked-prefill scoring on the GPU (MFMA path) against the CPU oracle (R:314-340)."""
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


def _case(count, prefix_len, seed, slots=20000):
    g = torch.Generator().manual_seed(seed)
    b = backend(gen=g, slots=slots)
    st = ge.state(b)
    q = (torch.randn((count, 64, 64), generator=g) * 1.5).to(torch.bfloat16).cuda()
    sinks = torch.randn(64, generator=g).to(torch.bfloat16).cuda()
    perm = torch.randperm(slots - 1, generator=g)[:prefix_len + count] + 1
    return b, st, q, sinks, perm[:prefix_len].cuda(), perm[prefix_len:].cuda()


@pytest.mark.parametrize("count,prefix_len,mode,delay", [
    (1, 0, 1, 0), (37, 0, 2, 0), (100, 300, 1, 0), (257, 1000, 2, 0), (130, 64, 1, 0),
    # Score delays (block policies): pass 2 credits keys `delay` positions older than each query
    # only, while pass 1's normaliser covers the whole causal range.
    (257, 1000, 2, 128), (130, 64, 1, 100), (37, 0, 1, 5), (200, 0, 2, 190), (20, 30, 1, 60)])
def test_prefill_scores_match_oracle(count, prefix_len, mode, delay):
    b, st, q, sinks, prefix, new = _case(count, prefix_len, seed=count + prefix_len)
    keys = b.token_to_kv_pool.get_key_buffer(1)
    before = torch.rand(st.scores.shape, generator=torch.Generator().manual_seed(3)).cuda()
    st.scores.copy_(before)
    ge._prefill_scores(st, 0, mode | delay << 8, layer(1), q, keys, sinks, prefix, new)
    upd, slots = O.prefill_score_update(mode, q.float().cpu().numpy(), keys.float().cpu().numpy(),
                                        sinks.float().cpu().numpy(), 0.125, 8, prefix.cpu().numpy(),
                                        new.cpu().numpy(), delay=delay)
    expected = before.clone()
    expected[0][:, torch.tensor(slots).cuda()] += torch.tensor(upd, dtype=torch.float32).cuda()
    torch.testing.assert_close(st.scores, expected, rtol=1e-3, atol=1e-6)


def _exact_scores(mode, q, keys, sinks, slots, prefix_len):
    """[KV head, list entry] column sums or maxima of the exact probabilities, in 64 bits."""
    count, total = q.shape[0], slots.numel()
    hidden = torch.arange(total, device="cuda") > prefix_len + torch.arange(count, device="cuda")[:, None]
    out = torch.zeros((8, total), dtype=torch.float64, device="cuda")
    for g in range(8):
        qg = q[:, 8 * g:8 * g + 8].double().transpose(0, 1)
        x = (torch.matmul(qg, keys[slots, g].double().t().contiguous()) * 0.125).masked_fill(hidden, -torch.inf)
        sink = sinks[8 * g:8 * g + 8].double().view(8, 1, 1)
        p = torch.exp(x - torch.logaddexp(torch.logsumexp(x, -1, keepdim=True), sink))
        out[g] = p.sum((0, 1)) if mode == 1 else p.amax(0).sum(0)
    return out


# Edges of the query blocks (8 per wave, 64 per workgroup), of the 64-key tiles and of the key
# ranges (4 tiles or more), and logits that move a row's reference: by a factor over 2^6 from tile
# to tile (scale 3), and past 2^64 (scale 40).
@pytest.mark.parametrize("mode", [1, 2])
@pytest.mark.parametrize("count,prefix_len,scale", [
    (1, 255, 1), (1, 256, 1), (7, 0, 1), (8, 63, 1), (9, 64, 1), (63, 449, 1), (64, 512, 1), (65, 1, 1),
    (129, 3000, 1), (513, 700, 1), (2, 9000, 1), (70, 1500, 3), (70, 1500, 40)])
def test_prefill_scores_at_the_edges_of_tiles_and_ranges(count, prefix_len, scale, mode):
    b, st, q, sinks, prefix, new = _case(count, prefix_len, seed=7 * count + prefix_len)
    keys = b.token_to_kv_pool.get_key_buffer(1)
    slots = torch.cat((prefix, new)).long()
    # Keys grow along the list, so later tiles hold larger logits.
    ramp = torch.linspace(0.1, scale, slots.numel(), device="cuda")[:, None, None]
    keys[slots] = (keys[slots].float() * ramp).to(keys.dtype)
    st.scores.zero_()
    ge._prefill_scores(st, 0, mode, layer(1), q, keys, sinks, prefix, new)
    want = _exact_scores(mode, q, keys, sinks, slots, prefix_len)
    # 32-bit logits: an absolute error of |x| * 2^-22 (64 products) is a relative error of p.
    largest = 1.5 * 8 * scale * 0.125 * 8 * 8
    torch.testing.assert_close(st.scores[0][:, slots].double(), want, rtol=1e-5 + largest * 2 ** -22, atol=1e-7)


# Both sides of pass 2's query-block rules: shorter blocks while few workgroups have work (60 and 850
# queries, not 1000), and longer ones in one round instead of a part of a second (2047, 1000 after
# 2500; 300 after 9000 would not fill it).
@pytest.mark.parametrize("mode", [1, 2])
@pytest.mark.parametrize("count,prefix_len", [(60, 0), (850, 0), (1000, 0), (780, 300), (2047, 0), (1000, 2500),
                                              (300, 9000)])
def test_prefill_scores_by_query_block_rule(count, prefix_len, mode):
    test_prefill_scores_at_the_edges_of_tiles_and_ranges(count, prefix_len, 1, mode)


@pytest.mark.parametrize("count,prefix_len", [(300, 0), (1000, 2500), (500, 9000)])
def test_normalisers_are_rounded_once(count, prefix_len):
    """A column sums thousands of rows' probabilities. One rounding of each normaliser (at most 2^-21
    in log2 units here) is as often up as down and all but cancels in it, as the exponentials' do, so
    what is left lies below 2^-23 in relative 2-norm; a logarithm with an error of its own does not
    cancel (2e-7)."""
    b, st, q, sinks, prefix, new = _case(count, prefix_len, seed=41)
    keys = b.token_to_kv_pool.get_key_buffer(1)
    slots = torch.cat((prefix, new)).long()
    st.scores.zero_()
    ge._prefill_scores(st, 0, 1, layer(1), q / 1.5, keys, sinks, prefix, new)
    want = _exact_scores(1, q / 1.5, keys, sinks, slots, prefix_len)
    got = st.scores[0][:, slots].double()
    assert float((got - want).norm() / want.norm()) < 2 ** -23


# The hooks build 32-bit slot lists; the entry also takes 64-bit ones, for every kind (sums, maxima,
# block counters of 4 keys 100 entries late) and more than one key range.
@pytest.mark.parametrize("mode", [1, 2, 4 | 2 << 4 | 100 << 8])
@pytest.mark.parametrize("count,prefix_len", [(70, 1500), (513, 0)])
def test_prefill_scores_of_64_bit_slot_lists(count, prefix_len, mode):
    from gstar_evict import _native as N
    b, st, q, sinks, prefix, new = _case(count, prefix_len, seed=31)
    keys = b.token_to_kv_pool.get_key_buffer(1)
    ws = torch.empty(N.lib().gse_prefill_workspace_bytes(count, 64), dtype=torch.uint8, device="cuda")
    got = []
    for slots in (torch.cat((prefix, new)).int(), torch.cat((prefix, new)).long()):
        sc = torch.zeros_like(st.scores[0])
        N.call("gse_prefill_scores", N.ptr(q), q.stride(0), q.stride(1), count, N.ptr(keys), keys.stride(0),
               keys.stride(1), N.ptr(slots), N.idx_code(slots), slots.numel(), prefix_len, N.ptr(sinks),
               N.float_code(sinks), mode, N.ptr(sc), sc.stride(0), sc.stride(1), 64, 8, 64, 0.125, N.ptr(ws),
               ws.numel(), N.stream())
        got.append(sc)
    assert float(got[0].sum()) > 0
    # The same sums, added in another order by the atomics: at most 2^-24 of the sum for each of the
    # query blocks (one per 32 queries at most).
    torch.testing.assert_close(got[1], got[0], rtol=17 * 2 ** -24, atol=0)


@pytest.mark.parametrize("n,m,first,second", [
    (0, 1, torch.int32, torch.int64), (255, 1, torch.int32, torch.int64), (1, 256, torch.int64, torch.int32),
    (300, 0, torch.int64, torch.int64), (257, 513, torch.int16, torch.int32)])
def test_visible_slots_of_any_index_width(n, m, first, second):
    from gstar_evict import attention
    prefix = torch.arange(3, 3 + 2 * n, 2, device="cuda").to(first)
    new = torch.arange(10 * m, 0, -5, device="cuda").to(second)[::2]  # a strided view
    got = attention.visible_slots(prefix, new)
    assert got.dtype == torch.int32
    assert got.tolist() == prefix.tolist() + new.tolist()


@pytest.mark.parametrize("ranges", [1, 2, 5])
def test_a_smaller_workspace_takes_fewer_key_ranges(ranges, monkeypatch):
    """The normalisers' bytes alone are enough; each further range of pass 1 adds its pairs."""
    count, prefix_len = 70, 3000
    b, st, q, sinks, prefix, new = _case(count, prefix_len, seed=9)
    keys = b.token_to_kv_pool.get_key_buffer(1)
    slots = torch.cat((prefix, new)).long()
    rows = count * 64
    size = -(-rows * 4 // 256) * 256 + (rows * 8 * ranges if ranges > 1 else 0)
    monkeypatch.setattr(st, "workspace", lambda name, nbytes: torch.empty(size, dtype=torch.uint8, device="cuda"))
    st.scores.zero_()
    ge._prefill_scores(st, 0, 1, layer(1), q, keys, sinks, prefix, new)
    want = _exact_scores(1, q, keys, sinks, slots, prefix_len)
    torch.testing.assert_close(st.scores[0][:, slots].double(), want, rtol=1e-4, atol=1e-7)


def test_after_extend_scores_chunks_of_two_requests():
    """The hook path: CSR prefix per request, zeroed new slots, sum and max rows in one batch."""
    g = torch.Generator().manual_seed(21)
    b = backend(gen=g)
    st = ge.state(b)
    perm = (torch.randperm(19999, generator=g) + 1).cuda()
    # Request rows 1 (head_sum, prefix 200, 50 new) and 2 (head_max_sum, prefix 0, 70 new).
    pre1, new1 = perm[:200], perm[200:250]
    pre2, new2 = perm[300:300], perm[300:370]
    for row, mode in ((1, 1), (2, 2)):
        st.entries[row] = {"kind": "live", "error": None, "mode": mode}
    q = torch.randn((120, 64, 64), generator=g).to(torch.bfloat16).cuda()
    sinks = torch.randn(64, generator=g).cuda()
    b.forward_metadata = SimpleNamespace(qo_indptr=torch.tensor([0, 50, 120], device="cuda"),
                                         kv_indptr=torch.tensor([0, 200, 200], device="cuda"),
                                         kv_indices=torch.cat((pre1, pre2)))
    fb = SimpleNamespace(req_pool_indices=torch.tensor([1, 2], device="cuda"),
                         out_cache_loc=torch.cat((new1, new2)), extend_prefix_lens_cpu=[200, 0])
    st.scores.fill_(0.5)
    ge.after_extend(b, q.reshape(120, -1), layer(1), fb, sinks)
    keys = b.token_to_kv_pool.get_key_buffer(1).float().cpu().numpy()
    expected = torch.full_like(st.scores, 0.5)
    expected[:, :, torch.cat((new1, new2))] = 0.0
    for (pre, new, lo, hi, mode) in ((pre1, new1, 0, 50, 1), (pre2, new2, 50, 120, 2)):
        upd, slots = O.prefill_score_update(mode, q[lo:hi].float().cpu().numpy(), keys, sinks.cpu().numpy(), 0.125,
                                            8, pre.cpu().numpy(), new.cpu().numpy())
        expected[0][:, torch.tensor(slots).cuda()] += torch.tensor(upd, dtype=torch.float32).cuda()
    torch.testing.assert_close(st.scores, expected, rtol=1e-3, atol=1e-6)


def test_prefill_mass_is_conserved_at_8k_chunk():
    """A full 8192-query chunk after a 2048-key prefix: head-sum scores of a KV head add up to the
    non-sink probability mass of its 8 query heads over all queries (a size-independent check)."""
    count, prefix_len = 8192, 2048
    b, st, q, sinks, prefix, new = _case(count, prefix_len, seed=5, slots=12000)
    keys = b.token_to_kv_pool.get_key_buffer(1)
    st.scores.zero_()
    ge._prefill_scores(st, 0, 1, layer(1), q, keys, sinks, prefix, new)
    got = st.scores[0].double().sum(1)  # [kv head]
    # Sink mass per (query, head) from the oracle on a sample of queries, exact elsewhere by sum.
    kk = keys[torch.cat((prefix, new))].float()
    total = torch.zeros(8, dtype=torch.float64)
    for lo in range(0, count, 1024):
        hi = lo + 1024
        qq = q[lo:hi].float().view(hi - lo, 8, 8, 64)
        logits = torch.einsum("qgjd,kgd->gjqk", qq, kk) * 0.125
        pos = prefix_len + torch.arange(lo, hi, device="cuda")
        logits.masked_fill_(torch.arange(kk.shape[0], device="cuda")[None, None, None, :] > pos[None, None, :, None],
                            -torch.inf)
        lse = torch.logsumexp(logits, -1)
        norm = torch.logaddexp(lse, sinks.float().view(8, 8, 1))
        sink_p = torch.exp(sinks.float().view(8, 8, 1) - norm)
        total += (1 - sink_p).sum((1, 2)).double().cpu()
    torch.testing.assert_close(got.cpu(), total, rtol=1e-4, atol=1e-3)


def test_index_reads_of_two_threads_do_not_meet(monkeypatch):
    """A second thread reads its vectors between the first one's wait and its copy to lists: each
    gets its own values."""
    import threading
    from concurrent.futures import ThreadPoolExecutor
    st = ge.state(backend())
    mine = [torch.tensor([3, 1], device="cuda"), torch.tensor([0, 5, 9], dtype=torch.int32, device="cuda")]
    other = [torch.tensor([7, 8], device="cuda"), torch.tensor([0, 2, 4], dtype=torch.int32, device="cuda")]
    stream_of, main, read = torch.cuda.current_stream, threading.current_thread(), []
    with ThreadPoolExecutor(1) as pool:
        def current_stream(device=None):
            stream = stream_of(device)

            def synchronize():
                stream.synchronize()
                if threading.current_thread() is main:
                    read.append(pool.submit(st.read_ints, *other).result())
            return SimpleNamespace(synchronize=synchronize)
        monkeypatch.setattr(torch.cuda, "current_stream", current_stream)
        assert st.read_ints(*mine) == [[3, 1], [0, 5, 9]]
    assert read == [[[7, 8], [0, 2, 4]]]
