"""The decode step as one native call against the same step op by op: hidden states, every pool and the context counters."""

import pytest
import torch

from _util import cpu_gen, same_bits

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def config(**kw):
    from isoexec_amd.runtimes.hybrid import HybridConfig

    base = dict(hidden=512, vocab=1024, layers=4, attention_every=2, gdn_k_heads=2, gdn_v_heads=4, q_heads=4, kv_heads=2,
                experts=16, topk=4, expert_inter=256, max_positions=256)
    return HybridConfig(**{**base, **kw})


def pools(engine):
    for i, g in engine.gdn.items():
        for name in ("ssm_state", "conv_state", "last_used", "_clock"):
            yield f"gdn {i} {name}", getattr(g, name)
    for i, kv in engine.kv.items():
        yield f"keys {i}", kv.k
        yield f"values {i}", kv.v


@pytest.mark.parametrize("n,kw", [
    (1, {}), (5, {}), (70, {}), (300, {}),                           # one-launch routing up to 256 tokens, packed dense up to 64
    (3, dict(hidden=2048, topk=8, experts=128, expert_inter=512)),
    (4, dict(experts=200, topk=2, hidden=2048)),                     # more experts than the one-launch routing holds
    (6, dict(moe_combine_dtype="bf16", attention_every=4)),
])
@pytest.mark.parametrize("packed", [True, False])
def test_native_step_equals_the_step_op_by_op(n, kw, packed):
    from isoexec_amd.runtimes.hybrid import HybridWeights, RolloutEngine

    cfg = config(**kw)
    w = HybridWeights.make(cfg, seed=3, device=DEV)
    g = cpu_gen(n)
    lens = [1 + (7 * i) % 11 for i in range(n)]
    tokens = torch.randint(0, cfg.vocab, (sum(lens),), generator=g).to(DEV)
    engines = [RolloutEngine(cfg, w, max_num_seqs=n, max_len=32, pack_expert_weights=packed) for _ in range(2)]
    slots = [(5 * i + 2) % 1021 for i in range(n)]
    for e in engines:
        e.prefill(slots, tokens, lens)
    one, ops = engines
    for step in range(3):
        tok = torch.randint(0, cfg.vocab, (n,), generator=g).to(DEV)
        ops.blocks.routing_log = []          # the log wants every layer's routing: op by op
        want = ops.decode(slots, tok)
        assert len(ops.blocks.routing_log) == cfg.layers
        got = one.decode(slots, tok)
        assert same_bits(got, want), step
        for (name, a), (_, b) in zip(pools(one), pools(ops)):
            assert torch.equal(a.reshape(-1).view(torch.uint8), b.reshape(-1).view(torch.uint8)), (step, name)
    # a captured step replays the native call: counters advance on the device, a replaced weight is seen by the next eager step
    graph = one.capture_decode(slots)
    ops.blocks.routing_log = None
    for step in range(3):
        tok = torch.randint(0, cfg.vocab, (n,), generator=g).to(DEV)
        ops.blocks.routing_log = []
        want = ops.decode(slots, tok)
        assert same_bits(graph.step(tok), want), step
        assert graph.state["ctx"].tolist() == [one.context[s] for s in slots]


def test_the_step_without_the_cache_extent_gives_the_same_bits():
    """``ix_decode_step``, for callers that keep positions in range themselves, against the checked form."""
    from isoexec_amd import _lib
    from isoexec_amd.runtimes.hybrid import HybridWeights, RolloutEngine

    cfg = config()
    w = HybridWeights.make(cfg, seed=7, device=DEV)
    one, plain = (RolloutEngine(cfg, w, max_num_seqs=2, max_len=32) for _ in range(2))
    tok = torch.tensor([5, 6], device=DEV)
    for e in (one, plain):
        e.prefill([0, 1], torch.tensor([1, 2, 3], device=DEV), [2, 1])
    want = one.decode([0, 1], tok)
    dims, layers = plain._native_step_tables(2)
    st, b = plain._decode_state([0, 1]), plain.blocks
    need = _lib.lib().ix_decode_step_workspace_bytes(dims.buffer_info()[0])
    work = torch.empty(need, dtype=torch.uint8, device=DEV)
    out = torch.empty(2, cfg.hidden, dtype=torch.bfloat16, device=DEV)
    rc = _lib.lib().ix_decode_step(
        dims.buffer_info()[0], layers.buffer_info()[0], w.embed.data_ptr(), w.layers[0]["pre_norm"].data_ptr(),
        b.cos.data_ptr(), b.sin.data_ptr(), tok.data_ptr(), st["slots_t"].data_ptr(), st["ctx"].data_ptr(),
        st["kv_start"].data_ptr(), float(cfg.eps), work.data_ptr(), need, out.data_ptr(), _lib.current_stream(out.device))
    assert rc == _lib.IX_OK and same_bits(out, want) and st["ctx"].tolist() == [3, 2]
    for (name, a), (_, c) in zip(pools(plain), pools(one)):
        assert torch.equal(a.reshape(-1).view(torch.uint8), c.reshape(-1).view(torch.uint8)), name


def test_native_step_is_taken_and_sees_replaced_weights():
    from isoexec_amd.runtimes.hybrid import HybridWeights, RolloutEngine

    cfg = config()
    w = HybridWeights.make(cfg, seed=4, device=DEV)
    e = RolloutEngine(cfg, w, max_num_seqs=2, max_len=32)
    e.prefill([0, 1], torch.tensor([1, 2, 3], device=DEV), [2, 1])
    tok = torch.tensor([5, 6], device=DEV)
    st = e._decode_state([0, 1])
    first = e._decode_native(st, tok)
    assert first is not None and st["ctx"].tolist() == [3, 2]
    # tables are built per call: another norm weight, then a tensor the call cannot take (strided), which goes op by op
    w.final_norm = w.final_norm + 1.0
    moved = e._decode_native(e._decode_state([0, 1]), tok)
    assert moved is not None and not same_bits(moved, first)
    w.layers[0]["out_proj"] = torch.cat([w.layers[0]["out_proj"]] * 2, dim=1)[:, : cfg.gdn_z]
    assert e._decode_native(e._decode_state([0, 1]), tok) is None
    assert torch.isfinite(e.decode([0, 1], tok).float()).all()


@pytest.mark.parametrize("layer,name,cut", [(0, "out_proj", lambda w: w[:, :-8]), (0, "in_proj", lambda w: w[:-8]),
                                            (1, "o_proj", lambda w: w[:, :-8]), (1, "qkv_proj", lambda w: w[:-8]),
                                            (None, "embed", lambda w: w[:-8])])
def test_a_weight_of_another_shape_is_not_handed_to_the_native_step(layer, name, cut):
    from isoexec_amd.runtimes.hybrid import HybridWeights, RolloutEngine

    w = HybridWeights.make(config(), seed=4, device=DEV)
    e = RolloutEngine(config(), w, max_num_seqs=2, max_len=32)
    assert e._native_step_tables(2) is not None
    if layer is None:
        setattr(w, name, cut(getattr(w, name)).contiguous())
    else:
        w.layers[layer][name] = cut(w.layers[layer][name]).contiguous()
    assert e._native_step_tables(2) is None


def test_the_row_lookup_switch_sends_the_step_op_by_op(monkeypatch):
    from isoexec_amd.ops.gdn import gdn_cpr_rows
    from isoexec_amd.runtimes.hybrid import HybridWeights, RolloutEngine

    w = HybridWeights.make(config(), seed=6, device=DEV)
    engines = [RolloutEngine(config(), w, max_num_seqs=2, max_len=32) for _ in range(2)]
    tok = torch.tensor([5, 6], device=DEV)
    for e in engines:
        e.prefill([0, 1], torch.tensor([1, 2, 3], device=DEV), [2, 1])
    want = engines[0].decode([0, 1], tok)
    monkeypatch.setenv("SKYRL_ISOEXEC_GDN_CPR_FUSED_ROWS", "0")
    assert engines[1]._native_step_tables(2) is None
    served = gdn_cpr_rows._served
    got = engines[1].decode([0, 1], tok)
    assert gdn_cpr_rows._served == served and same_bits(got, want)
    for (name, a), (_, b) in zip(pools(engines[1]), pools(engines[0])):
        assert torch.equal(a.reshape(-1).view(torch.uint8), b.reshape(-1).view(torch.uint8)), name


@pytest.mark.parametrize("what", ["keys", "values", "ssm_state", "conv_state", "last_used", "slot2row", "sin", "cos", "experts"])
def test_a_pool_table_or_copy_of_another_shape_is_not_handed_to_the_native_step(what):
    """The kernels index these with what the pools' own tables say: a tensor of another shape, or of another type, goes op by
    op, where the ops' own checks refuse it."""
    from isoexec_amd.runtimes.hybrid import HybridWeights, RolloutEngine

    cfg = config(expert_inter=512)
    e = RolloutEngine(cfg, HybridWeights.make(cfg, seed=4, device=DEV), max_num_seqs=2, max_len=32)
    assert e._native_step_tables(2) is not None
    if what in ("keys", "values"):
        kv, name = e.kv[1], what[0]
        setattr(kv, name, getattr(kv, name)[:, :16].contiguous())
    elif what in ("sin", "cos"):
        setattr(e.blocks, what, getattr(e.blocks, what).float())
    elif what == "experts":
        w1f, w2f = e.blocks.packed_experts[2]
        e.blocks.packed_experts[2] = (w1f[:-1].contiguous(), w2f)
    else:
        g = e.gdn[0]
        setattr(g, what, getattr(g, what)[:-1].contiguous())
    assert e._native_step_tables(2) is None
    if what == "experts":
        with pytest.raises(RuntimeError, match="pack_decode"):
            e.blocks.moe(2, torch.zeros(2, 512, dtype=torch.bfloat16, device=DEV))


@pytest.mark.parametrize("captured", [False, True])
@pytest.mark.parametrize("field,value", [("ctx", 32), ("ctx", -1), ("ctx", 2**31 - 2), ("kv_start", 4 * 32), ("kv_start", -32),
                                         ("kv_start", 4 * 32 - 2), ("kv_start", 2**62), ("token", 1024), ("token", -1),
                                         ("token", 2**62)])
def test_a_position_or_token_out_of_range_stores_nothing_and_is_reported(field, value, captured):
    """The step's own counters can run past what the host's bookkeeping says. Sequence 1 of 3 gets a position (or a first cache
    token) that does not fit the 4 x 32 tokens of the cache, or a token id that the vocabulary of 1024 does not hold: its
    output is NaN, no pool changes for it, the others' bits are those of the untouched step, and the next call raises."""
    from isoexec_amd.runtimes.hybrid import HybridWeights, RolloutEngine

    cfg = config()
    w = HybridWeights.make(cfg, seed=5, device=DEV)
    e, ref = (RolloutEngine(cfg, w, max_num_seqs=3, max_len=32) for _ in range(2))
    tok = torch.tensor([5, 6, 7], device=DEV)
    for engine in (e, ref):
        engine.prefill([0, 1, 2], torch.tensor([1, 2, 3, 4, 5], device=DEV), [2, 1, 2])
        engine.decode([0, 1, 2], tok)
    row = e.kv_rows[1]
    before = {name: t.clone() for name, t in pools(e)}
    st, given = e._decode_state([0, 1, 2]), tok.clone()
    if captured:
        graph = e.capture_decode([0, 1, 2])
        st = graph.state
    (given if field == "token" else st[field])[1] = value
    out = graph.step(given).clone() if captured else e._decode_native(st, given)
    want = ref.decode([0, 1, 2], tok)
    assert out[1].isnan().all() and same_bits(out[[0, 2]], want[[0, 2]])
    for (name, got), (_, other) in zip(pools(e), pools(ref)):
        if name.endswith(("last_used", "_clock")):
            continue
        r = e.gdn[0].table.row_of[1] if name.startswith("gdn") else row
        keep = [i for i in range(1, 4) if i != r]  # row 0 is the null row
        assert torch.equal(got[r], before[name][r]) and torch.equal(got[keep], other[keep]), name
    with pytest.raises(RuntimeError, match="outside the vocabulary" if field == "token" else "outside its part"):
        graph.step(tok) if captured else e.decode([0, 1, 2], tok)
    e.check_steps()  # reported once
