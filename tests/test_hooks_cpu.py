"""The scheduler hooks' refusals, on CPU tensors (no kernel runs): invalid configs, retracted
requests, chunks that rewind below the frontier or cross a 2048 boundary, and rows that change
hands. Each turns the request inert with the reference's error text and policy mode 0
(R:625-637, R:640-689); a retraction also writes its payload (R:668-674)."""
import sys
import types
from types import SimpleNamespace

import pytest
import torch

from fakes import backend


@pytest.fixture
def hooks(monkeypatch, tmp_path):
    monkeypatch.setenv("GSTAR_PAYLOAD_DIR", str(tmp_path))
    names = ["sglang", "sglang.srt", "sglang.srt.mem_cache", "sglang.srt.mem_cache.unified_cache",
             "sglang.srt.mem_cache.unified_cache.component_type"]
    for name in names:
        monkeypatch.setitem(sys.modules, name, types.ModuleType(name))
    sys.modules[names[-1]].ComponentType = SimpleNamespace(SWA="swa")
    import gstar_evict
    gstar_evict.STATE = None
    gstar_evict.RETRACTED.clear()
    st = gstar_evict.state(backend(rows=4, width=8192, slots=64, layers=2, full=(0,), device="cpu"))
    yield gstar_evict, st, tmp_path
    gstar_evict.STATE = None
    gstar_evict.RETRACTED.clear()


CFG = {"name": "head_sum_2048", "budget": 2048, "prefix": 128, "recent": 512, "seed": 0}


def _req(rid, row, start, length, params=None, retraction=0):
    return SimpleNamespace(rid=rid, session=None, retraction_count=retraction,
                           sampling_params=SimpleNamespace(custom_params=params),
                           extend_range=SimpleNamespace(start=start, length=length),
                           kv=SimpleNamespace(req_pool_idx=row, get_evicted_seqlen=lambda kind: 0))


def _extend(ge, *reqs):
    ge.on_extend(SimpleNamespace(reqs=list(reqs), tree_cache=SimpleNamespace(token_to_kv_pool_allocator=None)))


def test_valid_config_gets_a_mode_and_a_fresh_row(hooks):
    ge, st, _ = hooks
    st.frontier[1], st.count[1] = 77, 5  # stale state from a previous owner of the row
    _extend(ge, _req("a", 1, 0, 2048, {"gstar_eviction": CFG}))
    e = st.entries[1]
    assert e["error"] is None and e["kind"] == "live" and int(st.mode[1]) == 1
    assert int(st.frontier[1]) == 0 and int(st.count[1]) == 0


@pytest.mark.parametrize("cfg,message", [
    ({**CFG, "prefix": 2000}, "invalid gstar eviction settings"),          # P + R > B
    ({**CFG, "name": "lru_2048"}, "invalid gstar eviction settings"),       # unknown policy
    ({**CFG, "name": "prefix_sliding_2048"}, "Prefix Sliding requires B = P + R"),
    ({k: v for k, v in CFG.items() if k != "budget"}, "'budget'"),          # missing key
])
def test_invalid_config_runs_unevicted(hooks, cfg, message):
    ge, st, _ = hooks
    _extend(ge, _req("a", 1, 0, 2048, {"gstar_eviction": cfg}))
    e = st.entries[1]
    assert message in e["error"] and e["mode"] == 0 and int(st.mode[1]) == 0


def test_requests_without_params_get_no_entry(hooks):
    ge, st, _ = hooks
    _extend(ge, _req("a", 1, 0, 2048, None), _req("b", 2, 0, 2048, {"other": 1}))
    assert st.entries == {}


def test_retracted_request_is_refused_and_stays_refused(hooks):
    ge, st, tmp = hooks
    from gstar_evict import retention
    _extend(ge, _req("a", 1, 0, 2048, {"gstar_eviction": CFG}, retraction=1))
    e = st.entries[1]
    assert e["error"] == "retracted" and int(st.mode[1]) == 0 and "a" in ge.RETRACTED
    doc = retention.read_payload(tmp / "a-retracted.json.gz")
    assert doc["kind"] == "retracted" and doc["cfg"] == CFG
    # The same request on a fresh row (its key is remembered) is refused too.
    _extend(ge, _req("a", 2, 0, 2048, {"gstar_eviction": CFG}))
    assert st.entries[2]["error"] == "retracted" and int(st.mode[2]) == 0


def test_rewind_below_the_frontier_is_an_error(hooks):
    ge, st, _ = hooks
    _extend(ge, _req("a", 1, 0, 2048, {"gstar_eviction": CFG}))
    st.entries[1]["frontier"] = 4096  # as after a boundary at 4096
    _extend(ge, _req("a", 1, 2048, 1024, {"gstar_eviction": CFG}))
    assert st.entries[1]["error"] == "the session rewound below the eviction frontier"
    assert int(st.mode[1]) == 0


@pytest.mark.parametrize("start,length,ok", [(2000, 48, True), (2000, 49, False), (100, 1948, True),
                                             (4000, 200, False), (2049, 2047, True), (2049, 2048, False)])
def test_chunk_crossing_a_boundary_is_an_error(hooks, start, length, ok):
    ge, st, _ = hooks
    _extend(ge, _req("a", 1, start, length, {"gstar_eviction": CFG}))
    e = st.entries[1]
    if ok:
        assert e["error"] is None and int(st.mode[1]) == 1
    else:
        assert e["error"] == "prefill chunk crosses a boundary; use --chunked-prefill-size 2048"
        assert int(st.mode[1]) == 0


def test_errors_keep_the_row_inert_and_a_new_owner_starts_clean(hooks):
    ge, st, _ = hooks
    _extend(ge, _req("a", 1, 2000, 100, {"gstar_eviction": CFG}))
    assert st.entries[1]["error"]
    _extend(ge, _req("a", 1, 2100, 100, {"gstar_eviction": CFG}))  # later chunks: still refused
    assert st.entries[1]["error"] and int(st.mode[1]) == 0
    _extend(ge, _req("b", 1, 0, 2048, {"gstar_replay": CFG}))  # the row changes hands
    e = st.entries[1]
    assert e["key"] == "b" and e["kind"] == "replay" and e["error"] is None and int(st.mode[1]) == 1


def test_diagnostic_specs_take_their_own_protection(hooks):
    """T:240-244: each comma-separated spec keeps its own name, budget, prefix and recent."""
    ge, _, _ = hooks
    req = SimpleNamespace(rid="r", session=None, origin_input_ids=[0] * 10)
    e = ge._diagnostic_entry(req, {"policies": "random_2048:8192:2048:2048,prefix_sliding_2048:8192:2048:6144"},
                             "cpu", 12, 8)
    assert e["specs"] == [("random_2048", 8192, 2048, 2048), ("prefix_sliding_2048", 8192, 2048, 6144)]
    assert tuple(e["resident"].shape) == (2, 12, 8, 10) and bool(e["resident"].all())


# ------------------------------------------------------------- CSR check --

def test_csr_check_accepts_a_well_formed_csr():
    from gstar_evict.attention import check_csr
    check_csr(torch.tensor([0, 3, 3, 5], dtype=torch.int32), torch.tensor([1, 2, 3, 9, 4, 0, 0]), 3, 10)
    check_csr(torch.tensor([0], dtype=torch.int32), torch.zeros(0, dtype=torch.int32), 0, 10)


@pytest.mark.parametrize("indptr,indices,bs,slots,message", [
    ([0, 3], [1, 2, 3], 2, 10, "indptr has 2 entries"),
    ([1, 3, 5], [1, 2, 3, 4, 5], 2, 10, "indptr\\[0\\] is 1"),
    ([0, 4, 3], [1, 2, 3, 4], 2, 10, "decreases at sequence 1"),
    ([0, 3, 8], [1, 2, 3, 4, 5], 2, 10, "kv_indices holds 5"),
    ([0, 2, 4], [1, 2, 3, 10], 2, 10, "slot 10 outside the pool of 10"),
    ([0, 2, 4], [1, -2, 3, 4], 2, 10, "slot -2 outside"),
])
def test_csr_check_rejects_a_malformed_csr(indptr, indices, bs, slots, message):
    """The opt-in host check (GSTAR_EVICT_CHECK=1) names what is wrong with a decode CSR before any
    launch: a short indptr, a nonzero start, a decreasing offset, a list past kv_indices, a slot
    outside the pool."""
    from gstar_evict.attention import check_csr
    with pytest.raises(ValueError, match=message):
        check_csr(torch.tensor(indptr, dtype=torch.int32), torch.tensor(indices, dtype=torch.int32), bs, slots)


def test_csr_check_rejects_a_list_longer_than_max_len():
    """The launches size the score grids, the kept products and the fold's totals by max_len: a
    list longer than it is named (sequence 1 lists 5 keys against max_len 4); a list of exactly
    max_len keys passes."""
    from gstar_evict.attention import check_csr
    indptr, indices = torch.tensor([0, 3, 8], dtype=torch.int32), torch.tensor([1, 2, 3, 4, 5, 6, 7, 8])
    check_csr(indptr, indices, 2, 10, max_len=5)
    with pytest.raises(ValueError, match="sequence 1 lists 5 keys, more than max_len = 4"):
        check_csr(indptr, indices, 2, 10, max_len=4)


def test_csr_check_runs_before_the_decode_launch(hooks, monkeypatch):
    """With GSTAR_EVICT_CHECK=1 a malformed CSR raises in the decode hook, before the library is
    called (CPU tensors: a launch would fail differently)."""
    ge, st, _ = hooks
    st.check = True
    b = SimpleNamespace(forward_metadata=SimpleNamespace(kv_indptr=torch.tensor([0, 5], dtype=torch.int32),
                                                         kv_indices=torch.tensor([1, 2, 3], dtype=torch.int32)),
                        token_to_kv_pool=st.pool)
    lay = SimpleNamespace(tp_q_head_num=64, tp_k_head_num=8, qk_head_dim=64, layer_id=0, sliding_window_size=-1,
                          scaling=0.125)
    q = torch.zeros((1, 64 * 64), dtype=torch.bfloat16)
    from gstar_evict import attention
    with pytest.raises(ValueError, match="kv_indices holds 3"):
        attention.fused_decode(st, b, q, lay, SimpleNamespace(out_cache_loc=torch.zeros(1, dtype=torch.int64)),
                               torch.zeros(64), torch.zeros_like(q))


def test_a_batch_without_an_opted_in_row_needs_no_bounds(hooks):
    """after_extend of rows that opted out returns while another request is live, whatever its
    metadata holds; a batch with an opted-in row is refused without bounds."""
    from fakes import layer
    ge, st, _ = hooks
    _extend(ge, _req("a", 1, 0, 2048, {"gstar_eviction": CFG}))
    out = SimpleNamespace(req_pool_indices=torch.tensor([2, 3]))
    for b in (SimpleNamespace(), SimpleNamespace(forward_metadata=None),
              SimpleNamespace(forward_metadata=SimpleNamespace(qo_indptr=None)),
              SimpleNamespace(forward_metadata=SimpleNamespace(kv_indptr=torch.tensor([0, 5, 9])))):
        assert ge.after_extend(b, None, layer(0), out, None) is None
        with pytest.raises((ValueError, AttributeError)):
            ge.after_extend(b, None, layer(0), SimpleNamespace(req_pool_indices=torch.tensor([2, 1])), None)
