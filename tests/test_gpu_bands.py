"""Matrix products in bands of 96 .. 224 rows (pipeline G) against the other tiles, bit for bit: heights around the edges of a
band, the shortest K, ragged columns, the row maximum, and the calls a band is chosen for by size but does not serve."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _randn(*shape, seed, std=1.0):
    g = torch.Generator(device=DEV)
    g.manual_seed(seed)
    return (torch.randn(*shape, generator=g, device=DEV) * std).to(torch.bfloat16)


@pytest.mark.parametrize("band", [128, 160, 192, 224])
@pytest.mark.parametrize("n,k", [(264, 768), (2048, 832), (70000, 768)])  # one k-tile per slice, a runtime one, many turns
def test_dense_bands(band, n, k):
    from isoexec_amd.ops.mm.mm_hip import linear_nt

    w = _randn(n, k, seed=1, std=0.05)
    for m in (1, 31, band - 1, band, band + 1, 2 * band + 33):
        x = _randn(m, k, seed=m)
        want, want_top = linear_nt(x, w, tile=6, want_row_max=True)
        got, top = linear_nt(x, w, tile=10 + band // 32, want_row_max=True)
        assert torch.equal(got, want) and torch.equal(top, want_top), m
        assert torch.equal(linear_nt(x, w, tile=10 + band // 32), want), m


def test_a_band_chosen_by_size_serves_every_call():
    from isoexec_amd import _lib
    from isoexec_amd.ops.mm.mm_hip import linear_nt

    m, n, k = 300, 40000, 768
    assert _lib.lib().ix_gemm_bf16_n_tiles(m, n, k, 0) == 4 * ((n + 255) // 256)  # a band's parts
    x, w, bias = _randn(m, k, seed=2), _randn(n, k, seed=3, std=0.05), _randn(n, seed=4)
    for kw in ({}, {"bias": bias}, {"out_dtype": torch.float32}):
        want, want_top = linear_nt(x, w, tile=6, want_row_max=True, **kw)
        got, top = linear_nt(x, w, want_row_max=True, **kw)
        assert torch.equal(got, want) and torch.equal(top, want_top), kw
        assert torch.equal(linear_nt(x, w, **kw), want), kw
    assert linear_nt(x, w, bias, tile=15) is None  # asked for by number it declines
    with pytest.raises(RuntimeError):
        linear_nt(x[:, :-8], w[:, :-4])


@pytest.mark.parametrize("bm", [96, 160, 192, 224])
@pytest.mark.parametrize("t,e,hd,f", [(300, 8, 1024, 768), (1111, 8, 1024, 896), (37, 4, 2048, 768)])
def test_expert_bands(bm, t, e, hd, f):
    from isoexec_amd.ops.moe.moe_hip import experts_forward, permute

    x, w1, w2 = _randn(t, hd, seed=5), _randn(e, 2 * f, hd, seed=6, std=0.03), _randn(e, hd, f, seed=7, std=0.03)
    g = torch.Generator().manual_seed(t)
    idx = torch.stack([torch.randperm(e - 1, generator=g)[:2] for _ in range(t)]).to(torch.int32).to(DEV)  # the last: no rows
    prob = torch.rand(t, 2, generator=g).to(DEV)
    want, wi = experts_forward(x, w1, w2, permute(idx, prob, e, BM=32), return_inter=True)
    got, gi = experts_forward(x, w1, w2, permute(idx, prob, e, BM=bm), return_inter=True)
    assert torch.equal(gi, wi) and torch.equal(got, want)


def test_expert_bands_on_sizes_they_do_not_serve():
    from isoexec_amd.ops.moe.moe_hip import experts_forward, permute

    t, e, hd, f = 200, 4, 512, 320  # too few k-tiles, F not a multiple of 128
    x, w1, w2 = _randn(t, hd, seed=8), _randn(e, 2 * f, hd, seed=9, std=0.05), _randn(e, hd, f, seed=10, std=0.05)
    idx = torch.arange(2 * t, device=DEV, dtype=torch.int32).view(t, 2) % e
    prob = torch.rand(t, 2, device=DEV)
    want = experts_forward(x, w1, w2, permute(idx, prob, e, BM=32))
    assert torch.equal(experts_forward(x, w1, w2, permute(idx, prob, e, BM=160)), want)


def test_packed_matrices_of_another_layer_stay_refused_where_a_band_takes_over():
    from isoexec_amd.ops.moe.moe_hip import experts_forward, pack_decode, permute

    t, e, hd, f = 64, 4, 1024, 768  # 32 rows per expert
    x, w1, w2 = _randn(t, hd, seed=8), _randn(e, 2 * f, hd, seed=9, std=0.05), _randn(e, hd, f, seed=10, std=0.05)
    idx = torch.arange(2 * t, device=DEV, dtype=torch.int32).view(t, 2) % e
    p = permute(idx, torch.rand(t, 2, device=DEV), e, BM=96)
    w1f, w2f = pack_decode(w1, w2)
    assert torch.equal(experts_forward(x, w1, w2, p, packed=(w1f, w2f)), experts_forward(x, w1, w2, p))
    with pytest.raises(RuntimeError, match="pack_decode"):
        experts_forward(x, w1, w2, p, packed=(w1f[:2], w2f[:2]))
