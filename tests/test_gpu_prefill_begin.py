"""A prefill's table edits, use stamps and zeroed rows in one launch, against torch's operators."""

import pytest
import torch

from _util import cpu_gen, same_bits

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def layers(kind, capacity=4):
    g = cpu_gen(1)
    H, HV, K, V = 2, 4, 128, 128
    d = 2 * H * K + HV * V
    kw = dict(capacity=capacity, conv_weight=torch.randn(d, 4, generator=g).to(torch.bfloat16).to(DEV),
              conv_bias=torch.randn(d, generator=g).to(torch.bfloat16).to(DEV), A_log=torch.randn(HV, generator=g).to(DEV),
              dt_bias=torch.randn(HV, generator=g).to(DEV), num_k_heads=H, head_k_dim=K, num_v_heads=HV, head_v_dim=V, device=DEV)
    if kind == "native":
        kw.update(ssm_state=torch.full((capacity + 1, HV, V, K), 7.0, device=DEV),
                  conv_state=torch.zeros(capacity + 1, d, 3, dtype=torch.bfloat16, device=DEV))
    if kind == "cpr":
        from isoexec_amd.ops.gdn.gdn_cpr_state import CprGDN

        return CprGDN(**kw, chunk_size=16), d, HV
    from isoexec_amd.ops.gdn.gdn_recurrent_state import RecurrentGDN

    return RecurrentGDN(**{k: (v.clone() if kind == "native" and k.endswith("_state") else v) for k, v in kw.items()}), d, HV


@pytest.mark.parametrize("kind", ["own", "native", "cpr"])
def test_one_launch_leaves_what_the_operators_leave(kind, monkeypatch):
    monkeypatch.setenv("SKYRL_ISOEXEC_GDN_CHUNKED_PREFILL", "1")
    (one, d, hv), (ops, _, _) = layers(kind), layers(kind)
    assert one._begin_served(torch.device(DEV))
    monkeypatch.setattr(ops, "_begin_served", lambda dev: False)
    for layer in (one, ops):
        layer.ssm_state.fill_(3.0)
    g = cpu_gen(2)
    # new slots, a resumed one beside a new one, no fresh row, an empty sequence beside another, more slots than free rows (evictions)
    steps = [([1, 3], [5, 1], [False, False]), ([3, 2], [4, 17], [True, False]), ([1, 2], [2, 3], [True, True]),
             ([4, 1], [0, 3], [False, True])]
    if kind == "own":
        steps += [([900, 901, 902], [3, 1, 2], None), ([900, 5], [6, 2], [True, False])]
    for slots, lens, cont in steps:
        t = sum(lens)
        qsl = [sum(lens[:i]) for i in range(len(lens) + 1)]
        x = torch.randn(t, d, generator=g).to(torch.bfloat16).to(DEV)
        a, b = (torch.randn(t, hv, generator=g).to(torch.bfloat16).to(DEV) for _ in range(2))
        dev_slots = torch.tensor(slots, device=DEV)
        before = one.pos.clone() if kind == "cpr" else None
        out = [ly.prefill(dev_slots, slots, x, a, b, qsl, has_initial_state=cont) for ly in (one, ops)]
        assert same_bits(*out)
        names = ["ssm_state", "conv_state"] + ([] if kind == "native" else ["slot2row", "last_used", "_clock"])
        for name in names + (["entry_state", "pos"] if kind == "cpr" else []):
            assert torch.equal(getattr(one, name), getattr(ops, name)), (slots, name)
        for slot, n, resumed in zip(slots, lens, cont or []):
            if kind == "cpr":
                row = one.require_row(slot)
                assert one.pos[row] == n + (before[row] if resumed else 0)
    if kind == "native":
        assert (one.ssm_state[0] == 0).all()  # the null row


@pytest.mark.parametrize("kind", ["own", "cpr"])
def test_what_the_launch_resets_and_what_it_leaves(kind):
    """Resumed rows and rows of other slots keep their state and position, fresh ones and the null row lose them; a slot named twice
    has one row and its last stamp; evicted slots lead nowhere."""
    (one, _, _), (ops, _, _) = layers(kind), layers(kind)
    dev = torch.device(DEV)

    def both(slots, cont, qsl):
        got = one._prefill_begin(slots, None, cont, qsl, None, dev)
        rows = ops._assign_many(slots)
        want = (rows, *ops._prefill_upload(rows, cont, qsl, None, dev))
        assert got[0] == want[0] and all(torch.equal(g, w) for g, w in zip(got[1:], want[1:]))
        for name in ["ssm_state", "slot2row", "last_used", "_clock"] + (["entry_state", "pos"] if kind == "cpr" else []):
            assert torch.equal(getattr(one, name), getattr(ops, name)), name
        return got[0]

    def marked():
        for ly in (one, ops):
            ly.ssm_state.fill_(3.0)
            if kind == "cpr":
                ly.entry_state.fill_(5.0)
                ly.pos.fill_(7)

    kept = lambda r: bool((one.ssm_state[r] == 3.0).all()) and (kind != "cpr" or bool((one.entry_state[r] == 5.0).all()) and one.pos[r] == 7)
    zero = lambda r: bool((one.ssm_state[r] == 0.0).all()) and (kind != "cpr" or bool((one.entry_state[r] == 0.0).all()) and one.pos[r] == 0)
    a, b = both([1, 3], [False, False], [0, 2, 5])
    marked()
    (a2, c) = both([1, 2], [True, False], [0, 1, 4])
    assert a2 == a and kept(a) and kept(b) and zero(c) and zero(0)
    marked()
    d, d2, a3 = both([9, 9, 1], [False, False, False], [0, 2, 2, 3])  # one row left, named twice; a slot starts anew
    assert d == d2 and a3 == a and zero(d) and zero(a) and kept(b) and kept(c)
    assert one.last_used[d] == one._clock - 1 and one.last_used[a] == one._clock
    marked()
    e, f = both([50, 51], [False, False], [0, 1, 2])  # the pool is full: the two least recently used rows go
    assert {e, f} == {b, c} and one.slot2row[3] == 0 and one.slot2row[2] == 0 and zero(e) and zero(f) and kept(a) and kept(d)


def test_prefill_with_and_without_the_l2norm_in_the_convolution():
    (one, d, hv), (two, _, _) = layers("own"), layers("own")
    x = torch.randn(40, d, generator=cpu_gen(3)).to(torch.bfloat16).to(DEV)
    a = torch.randn(40, hv, generator=cpu_gen(4)).to(torch.bfloat16).to(DEV)
    slots = torch.tensor([1, 2], device=DEV)
    got = one.prefill(slots, [1, 2], x, a, a, [0, 23, 40])
    want = two.prefill(slots, [1, 2], x, a, a, [0, 23, 40], fuse_l2norm=False)
    assert same_bits(got, want) and same_bits(one.ssm_state, two.ssm_state) and same_bits(one.conv_state, two.conv_state)
