"""The 32 x 32 tile of the dense product (id 9) against the 64 x 32 one, whose bits are the oracle's."""

import pytest
import torch

from _util import cpu_gen, same_bits

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


# rows and columns around one and two tiles, fewer k-tiles than the ring holds, as many, one more, a K that ends inside a k-tile
@pytest.mark.parametrize("K", [8, 64, 200, 576, 640, 704, 4096])
@pytest.mark.parametrize("M,N", [(1, 32), (31, 33), (32, 2048), (33, 40), (64, 128), (65, 8), (257, 100)])
def test_tile_of_32_rows_and_columns(M, N, K):
    from isoexec_amd.ops.mm.mm_hip import linear_nt

    g = cpu_gen(M + N + K)
    x = torch.randn(M, K, generator=g).to(torch.bfloat16).to(DEV)
    w = torch.randn(N, K, generator=g).to(torch.bfloat16).to(DEV)
    bias = torch.randn(N, generator=g).to(torch.bfloat16).to(DEV)
    for dtype in (torch.bfloat16, torch.float32):
        want, want_top = linear_nt(x, w, tile=6, out_dtype=dtype, want_row_max=True)
        got, top = linear_nt(x, w, tile=9, out_dtype=dtype, want_row_max=True)
        assert same_bits(got, want) and same_bits(top, want_top)
        assert same_bits(linear_nt(x, w, tile=0, out_dtype=dtype), want)
        assert same_bits(linear_nt(x, w, bias, tile=9, out_dtype=dtype), linear_nt(x, w, bias, tile=6, out_dtype=dtype))


# the sizes at which the rule changes over (32 rows; 256 tiles), with the row maximum of the shape it takes
@pytest.mark.parametrize("M,N,K", [(32, 5120, 512), (33, 5120, 512), (64, 4096, 512), (65, 4096, 512), (128, 2048, 512), (129, 64, 512),
                                   (16, 32000, 2048), (17, 32000, 2048)])
def test_rule_of_the_small_tiles(M, N, K):
    from isoexec_amd.ops.mm.mm_hip import linear_nt

    g = cpu_gen(M + N)
    x = torch.randn(M, K, generator=g).to(torch.bfloat16).to(DEV)
    w = torch.randn(N, K, generator=g).to(torch.bfloat16).to(DEV)
    want, want_top = linear_nt(x, w, tile=6, want_row_max=True)
    got, top = linear_nt(x, w, want_row_max=True)
    assert same_bits(got, want) and same_bits(top, want_top)


# Weight rows 4 KiB apart, with and without a gap, and rows that only the row maximum's count takes for such (a gap, a bias): the
# columns of a last tile of 32 and of 128, the row maximum of every part that is counted.
@pytest.mark.parametrize("M,K,pitch", [(1, 2048, 2048), (16, 2048, 2048), (17, 2048, 2048), (7, 1984, 2048), (7, 2048, 2112)])
def test_few_rows_against_weight_rows_4_kib_apart(M, K, pitch):
    from isoexec_amd.ops.mm.mm_hip import linear_nt

    N = 80040
    g = torch.Generator(device=DEV)
    g.manual_seed(M + K + pitch)
    w = torch.randn(N, pitch, generator=g, device=DEV, dtype=torch.bfloat16)[:, :K]
    x = torch.randn(M, K, generator=g, device=DEV, dtype=torch.bfloat16)
    bias = torch.randn(N, generator=g, device=DEV, dtype=torch.bfloat16)
    for b in (None, bias):
        for dtype in (torch.bfloat16, torch.float32):
            want, want_top = linear_nt(x, w, b, tile=6, out_dtype=dtype, want_row_max=True)
            got, top = linear_nt(x, w, b, out_dtype=dtype, want_row_max=True)
            assert same_bits(got, want) and same_bits(top, want_top)
            assert same_bits(linear_nt(x, w, b, out_dtype=dtype), want)
