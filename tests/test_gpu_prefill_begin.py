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
    (one, d, hv), (ops, _, _) = layers(kind), layers(kind)
    assert one._begin_served(torch.device(DEV))
    monkeypatch.setattr(ops, "_begin_served", lambda dev: False)
    for layer in (one, ops):
        layer.ssm_state.fill_(3.0)
    g = cpu_gen(2)
    # new slots, a resumed one beside a new one, no fresh row, more slots than free rows (evictions), an empty sequence
    steps = [([1, 3], [5, 1], None), ([3, 2], [4, 17], [True, False]), ([1, 2], [2, 3], [True, True]), ([4], [0], None)]
    if kind == "own":
        steps += [([900, 901, 902], [3, 1, 2], None), ([900, 5], [6, 2], [True, False])]
    for slots, lens, cont in steps:
        t = sum(lens)
        qsl = [sum(lens[:i]) for i in range(len(lens) + 1)]
        x = torch.randn(t, d, generator=g).to(torch.bfloat16).to(DEV)
        a, b = (torch.randn(t, hv, generator=g).to(torch.bfloat16).to(DEV) for _ in range(2))
        dev_slots = torch.tensor(slots, device=DEV)
        if t:
            out = [ly.prefill(dev_slots, slots, x, a, b, qsl, has_initial_state=cont) for ly in (one, ops)]
            assert same_bits(*out)
        names = ["ssm_state", "conv_state"] + ([] if kind == "native" else ["slot2row", "last_used", "_clock"])
        for name in names + (["entry_state", "pos"] if kind == "cpr" else []):
            assert torch.equal(getattr(one, name), getattr(ops, name)), (slots, name)
    if kind == "native":
        assert (one.ssm_state[0] == 0).all()  # the null row


def test_prefill_with_and_without_the_l2norm_in_the_convolution():
    (one, d, hv), (two, _, _) = layers("own"), layers("own")
    x = torch.randn(40, d, generator=cpu_gen(3)).to(torch.bfloat16).to(DEV)
    a = torch.randn(40, hv, generator=cpu_gen(4)).to(torch.bfloat16).to(DEV)
    slots = torch.tensor([1, 2], device=DEV)
    got = one.prefill(slots, [1, 2], x, a, a, [0, 23, 40])
    want = two.prefill(slots, [1, 2], x, a, a, [0, 23, 40], fuse_l2norm=False)
    assert same_bits(got, want) and same_bits(one.ssm_state, two.ssm_state) and same_bits(one.conv_state, two.conv_state)
