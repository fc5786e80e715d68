"""Weights with one reader in a launch are read past the caches: the products on either side of that rule against a tile
that never takes it. Sums are the same in the same order, so every bit has to agree."""
import pytest
import torch

pytestmark = pytest.mark.gpu

@pytest.mark.parametrize("n, k", [(16384, 2048), (16376, 2048), (16640, 2112), (33000, 1024)])  # 64 MiB, just below, odd
@pytest.mark.parametrize("m, tile", [(1, 2), (127, 2), (128, 2), (129, 2), (129, 4), (256, 8), (257, 8)])
def test_dense(n, k, m, tile):
    from isoexec_amd.ops.mm.mm_hip import linear_nt

    g = torch.Generator(device="cuda")
    g.manual_seed(n + m)
    x = torch.randn(m, k, generator=g, device="cuda").to(torch.bfloat16)
    w = (0.02 * torch.randn(n, k, generator=g, device="cuda")).to(torch.bfloat16)
    got, top = linear_nt(x, w, tile=tile, want_row_max=True)
    want, want_top = linear_nt(x, w, tile=6, want_row_max=True)
    assert torch.equal(got, want) and torch.equal(top, want_top)

@pytest.mark.parametrize("tokens", [223, 224, 225, 449])  # mean rows per expert on either side of 224, a last row tile
def test_experts(tokens):
    from isoexec_amd.ops.moe import moe_hip as M

    # few experts; 704 output columns are 11 k-tiles of the second product, the fewest its streaming form takes
    e, h, f, k = 64, 1024, 768, 1
    g = torch.Generator(device="cuda")
    g.manual_seed(tokens)
    rows = tokens * e
    x = torch.randn(rows, h, generator=g, device="cuda").to(torch.bfloat16)
    w1 = (0.02 * torch.randn(e, 2 * f, h, generator=g, device="cuda")).to(torch.bfloat16)
    w2 = (0.02 * torch.randn(e, h, f, generator=g, device="cuda")).to(torch.bfloat16)
    idx, prob, _, _ = M.router_topk(torch.randn(rows, e, generator=g, device="cuda"), k, pre_softmax=True)
    got = M.experts_forward(x, w1, w2, M.permute(idx, prob, e, BM=256))
    want = M.experts_forward(x, w1, w2, M.permute(idx, prob, e, BM=128))
    assert torch.equal(got, want)
