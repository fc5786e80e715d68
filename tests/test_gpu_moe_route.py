"""Router and permutation at the edges of their splits -- lanes without experts, one and many waves of the expert scan, one
token and a full tile, every choice count -- against plain integer and fp32 arithmetic on the CPU."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _expect(logits, k, pre_softmax):
    x = torch.where(logits.isnan(), torch.full_like(logits, float("-inf")), logits)
    order = torch.argsort(x, dim=1, descending=True, stable=True)[:, :k]  # ties: the lowest expert
    top = torch.gather(x.double(), 1, order)
    p = torch.softmax(x.double(), 1).gather(1, order) if pre_softmax else torch.exp(top - top[:, :1])
    return order.int(), p / p.sum(1, keepdim=True)


def _check_permutation(p, idx, prob, E):
    T, k = idx.shape
    idx, prob = idx.cpu().long(), prob.cpu()
    counts = torch.bincount(idx.reshape(-1), minlength=E)
    offsets = torch.cat([torch.zeros(1, dtype=torch.long), counts.cumsum(0)])
    assert torch.equal(p.counts.cpu().long(), counts) and torch.equal(p.offsets.cpu().long(), offsets)
    flat = torch.argsort(idx.reshape(-1) * T + torch.arange(T).repeat_interleave(k))  # expert major, token ascending
    assert torch.equal(p.sorted_token.cpu().long(), flat // k)
    assert torch.equal(p.permuted_prob.cpu(), prob.reshape(-1)[flat])
    pos = torch.empty(T * k, dtype=torch.long)
    pos[flat] = torch.arange(T * k)
    by_expert = torch.argsort(idx, dim=1)
    assert torch.equal(p.combine_rows.cpu().long(), pos.reshape(T, k).gather(1, by_expert))
    n = int(p.tile_meta[0])
    tiles = p.tile_meta[1:].reshape(3, p.max_tiles)[:, :n].cpu().tolist()
    want = [(e, int(offsets[e]) + r, min(p.BM, int(counts[e]) - r)) for e in range(E) for r in range(0, int(counts[e]), p.BM)]
    assert list(zip(*tiles)) == want


@pytest.mark.parametrize("T", [1, 63, 64, 65, 256, 257])
@pytest.mark.parametrize("E, k", [(128, 8), (125, 8), (16, 16), (4, 1), (66, 2)])
@pytest.mark.parametrize("pre_softmax", [False, True])
def test_route(T, E, k, pre_softmax):
    from isoexec_amd.ops.moe import moe_hip as M

    g = torch.Generator().manual_seed(T * E)
    logits = torch.randn(T, E, generator=g).mul(4).round().div(4) if not pre_softmax else torch.randn(T, E, generator=g)
    logits[0, : E // 2] = float("nan") if E - E // 2 >= k else logits[0, : E // 2]
    logits[T // 2, E // 2 + 1:] = float("-inf") if E // 2 + 1 >= k else 0.0
    idx, prob, p = M.route_and_permute(logits.cuda(), k, pre_softmax=pre_softmax, BM=32)
    want_idx, want_p = _expect(logits, k, pre_softmax)
    assert torch.equal(idx.cpu(), want_idx)
    # exp to 2 ulp, a sum of at most 128 terms in a tree (7 roundings) and two divisions: below 16 * 2^-24 relative
    assert (prob.cpu().double() - want_p).abs().div(want_p + 1e-30).max() <= 16 * 2.0 ** -24
    _check_permutation(p, idx, prob, E)


@pytest.mark.parametrize("T, E, k", [(256, 512, 3), (200, 300, 16), (1000, 512, 5)])
def test_permute_many_experts(T, E, k):
    from isoexec_amd.ops.moe import moe_hip as M

    g = torch.Generator().manual_seed(E)
    idx = torch.argsort(torch.rand(T, E, generator=g), dim=1)[:, :k].int()
    prob = torch.rand(T, k, generator=g)
    _check_permutation(M.permute(idx.cuda(), prob.cuda(), E, BM=32), idx, prob, E)


def test_row_without_a_number():
    """An infinite logit makes a softmax row NaN: the choices stay valid, distinct experts."""
    from isoexec_amd.ops.moe import moe_hip as M

    logits = torch.randn(3, 128)
    logits[1, 7] = float("inf")
    idx, prob, _ = M.route_and_permute(logits.cuda(), 8, pre_softmax=True, BM=32)
    row = idx[1].cpu().tolist()
    assert len(set(row)) == 8 and min(row) >= 0 and max(row) < 128 and prob[1].isnan().all()
