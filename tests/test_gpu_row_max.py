"""The row maximum that a product's epilogue takes, where every value of a row is below zero: the columns past the matrix that
a tile pads with zeros are no part of it."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _positive(*shape, seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(seed)
    return (0.01 + torch.rand(*shape, generator=g, device=DEV)).to(torch.bfloat16)


@pytest.mark.parametrize("tile", [0, 1, 2, 4, 5, 6, 7, 8, 14, 15, 16, 17])
@pytest.mark.parametrize("n", [8, 64, 1024 + 64, 1024 + 128, 1024 + 136, 1024 + 200, 1024, 70000])  # 70000: many turns
def test_maximum_of_negative_products(tile, n):
    from isoexec_amd.ops.mm.mm_hip import linear_nt

    k = 768
    w = -_positive(n, k, seed=n)
    for m in (1, 65, 300):
        x = _positive(m, k, seed=m)
        x[m // 2, 5] = float("inf")  # a padded column of this row is inf * 0
        out, top = linear_nt(x, w, tile=tile, want_row_max=True)
        assert torch.equal(top, out.float().amax(1)) and float(top.max()) < 0.0, m


@pytest.mark.parametrize("rows", [7, 65, 129, 513])
def test_logprobs_of_rows_below_zero(rows):
    """The head's log-softmax with the product's maxima against the same logits through the maximum pass, at the vocabulary's
    593.5 tiles of 256 columns."""
    from isoexec_amd.ops.logprobs.rowinv import dense_head_logprobs, sampled_forward
    from isoexec_amd.ops.norms.fused_outnorm import fused_rms_norm_gamma
    from isoexec_amd.ops.mm.mm_hip import linear_nt
    from isoexec_amd.ops.logprobs.rowinv import leaves

    h, v = 2048, 151936
    hidden, head = _positive(rows, h, seed=rows), -_positive(v, h, seed=1)
    weight = torch.zeros(h, dtype=torch.bfloat16, device=DEV)
    target = torch.arange(rows, device=DEV) * 11
    got, logits = dense_head_logprobs(hidden, weight, head, target)
    x = fused_rms_norm_gamma(hidden, weight, 1e-6)
    assert torch.equal(logits, linear_nt(x, head))
    want, _ = sampled_forward(logits, target, leaves())
    assert torch.isfinite(want).all() and torch.equal(got, want)


# Sizes for which a band is chosen and does not serve the call; without bands the model takes the 256 x 256, 128 x 128 (odd
# number of its column tiles), 128 x 256 and 32 x 256 tile.
@pytest.mark.parametrize("m,n,k", [(138, 40696, 768), (148, 16920, 832), (4883, 776, 3584), (132, 19624, 1792)])
def test_shapes_that_take_a_bands_place(m, n, k):
    from isoexec_amd import _lib
    from isoexec_amd.ops.mm.mm_hip import linear_nt

    assert _lib.lib().ix_gemm_bf16_n_tiles(m, n, k, 0) == 4 * ((n + 255) // 256)
    x, w, bias = _positive(m, k, seed=2), -_positive(n, k, seed=3), -_positive(n, seed=4)
    for kw in ({"bias": bias}, {"out_dtype": torch.float32}):
        want, want_top = linear_nt(x, w, tile=6, want_row_max=True, **kw)
        got, top = linear_nt(x, w, want_row_max=True, **kw)
        assert torch.equal(got, want) and torch.equal(top, want_top), kw
