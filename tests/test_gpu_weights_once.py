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

@pytest.mark.parametrize("f", [704, 768])  # 11 k-tiles of the second product, the fewest its streaming form takes; and both streamed
@pytest.mark.parametrize("tokens", [223, 224, 225, 449])  # mean rows per expert on either side of 224, a last row tile
def test_experts(tokens, f):
    from isoexec_amd.ops.moe import moe_hip as M

    # few experts; five column tiles of the second product give its streaming form the 512 tiles it starts at
    e, h, k = 64, 1280, 1
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


MEMORY_SIDE_CACHE = 256 << 20  # the line of the packed streams


@pytest.mark.parametrize("m", [1, 32, 33, 64])
@pytest.mark.parametrize("n", [96, 65568])  # two and four waves per workgroup, a last unit without a neighbour
def test_packed_dense_on_either_side_of_the_line(m, n):
    from isoexec_amd import _lib
    from isoexec_amd.ops.mm.mm_hip import linear_nt, pack_nt_decode

    k = 1024
    g = torch.Generator(device="cuda")
    g.manual_seed(n + m)
    x = torch.randn(m, k, generator=g, device="cuda").to(torch.bfloat16)
    w = (0.02 * torch.randn(n, k, generator=g, device="cuda")).to(torch.bfloat16)
    wf = pack_nt_decode(w).packed
    want = linear_nt(x, w)
    for footprint in (0, MEMORY_SIDE_CACHE - 1, MEMORY_SIDE_CACHE):
        got = torch.full_like(want, float("nan"))
        rc = _lib.lib().ix_gemm_bf16_nt_decode_footprint(x.data_ptr(), k, wf.data_ptr(), got.data_ptr(), n, m, n, k, footprint,
                                                         _lib.current_stream(x.device))
        assert rc == _lib.IX_OK and torch.equal(got, want)


def test_a_step_op_by_op_says_what_its_dense_products_read(monkeypatch):
    """The products of a layer are below the line one by one; what decides is the model's packed weights together."""
    from isoexec_amd.runtimes.hybrid import HybridConfig, HybridWeights, RolloutEngine

    cfg = HybridConfig(hidden=1024, vocab=16384, layers=2, attention_every=2, gdn_k_heads=32, gdn_v_heads=32, q_heads=4,
                       kv_heads=2, experts=8, topk=2, expert_inter=128, max_positions=64, gdn_kernel="cpr")
    e = RolloutEngine(cfg, HybridWeights.make(cfg, seed=1, device="cuda:0"), max_num_seqs=1, max_len=32)
    packed = e.blocks.packed_dense
    total = sum(p.packed.numel() * 2 for p in packed.values())
    assert len(packed) == 2 and all(p.footprint == total > p.packed.numel() * 2 for p in packed.values())
    from isoexec_amd import _lib

    real, told = _lib.lib(), []

    class Told:
        def __getattr__(self, name):
            entry = getattr(real, name)
            if name != "ix_gemm_bf16_nt_decode_footprint":
                return entry
            return lambda *args: told.append(args[8]) or entry(*args)

    e.prefill([0], torch.tensor([1, 2], device="cuda:0"), [2])
    monkeypatch.setattr(_lib, "lib", Told)
    e.blocks.logits(e.decode([0], torch.tensor([3], device="cuda:0")))
    assert told == [total, total]


@pytest.mark.parametrize("bm, tokens", [(32, 1), (32, 33), (64, 33), (64, 130)])
def test_packed_experts_on_either_side_of_the_line(bm, tokens):
    from isoexec_amd import _lib
    from isoexec_amd.ops.moe import moe_hip as M

    e, h, f, k = 4, 512, 512, 2
    g = torch.Generator(device="cuda")
    g.manual_seed(tokens)
    x = torch.randn(tokens, h, generator=g, device="cuda").to(torch.bfloat16)
    w1 = (0.02 * torch.randn(e, 2 * f, h, generator=g, device="cuda")).to(torch.bfloat16)
    w2 = (0.02 * torch.randn(e, h, f, generator=g, device="cuda")).to(torch.bfloat16)
    w1f, w2f = M.pack_decode(w1, w2)
    idx, prob, _, _ = M.router_topk(torch.randn(tokens, e, generator=g, device="cuda"), k, pre_softmax=True)
    want = M.experts_forward(x, w1, w2, M.permute(idx, prob, e, BM=256))
    p = M.permute(idx, prob, e, BM=bm)
    for footprint in (0, MEMORY_SIDE_CACHE - 1, MEMORY_SIDE_CACHE):
        inter = torch.full((tokens * k, f), float("nan"), dtype=torch.bfloat16, device="cuda")
        got = torch.full_like(want, float("nan"))
        rc = _lib.lib().ix_moe_experts_packed_footprint(
            x.data_ptr(), h, p.sorted_token.data_ptr(), p.permuted_prob.data_ptr(), w1f.data_ptr(), w2f.data_ptr(),
            p.tile_meta.data_ptr(), p.max_tiles, bm, inter.data_ptr(), got.data_ptr(), tokens, tokens * k, h, f, footprint,
            _lib.current_stream(x.device))
        assert rc == _lib.IX_OK and torch.equal(got, want)
