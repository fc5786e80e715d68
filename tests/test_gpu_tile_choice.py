"""The tile shape the library chooses by itself, where its cost model moves from one shape to the next, against the
smallest tile asked for by name: same bits, and the row maxima laid out as the caller was told."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n, k", [(2048, 4096), (5120, 2048), (12352, 2048), (12352, 704), (20004, 1032)])
@pytest.mark.parametrize("m", [1, 65, 257, 384, 700, 1025])
@pytest.mark.parametrize("out_dtype", [torch.bfloat16, torch.float32])
def test_chosen_tile(m, n, k, out_dtype):
    from isoexec_amd.ops.mm.mm_hip import linear_nt

    g = torch.Generator(device="cuda")
    g.manual_seed(m)
    x = torch.randn(m, k, generator=g, device="cuda").to(torch.bfloat16)
    w = (0.02 * torch.randn(n, k, generator=g, device="cuda")).to(torch.bfloat16)
    got, top = linear_nt(x, w, out_dtype=out_dtype, want_row_max=True)
    want, want_top = linear_nt(x, w, out_dtype=out_dtype, tile=6, want_row_max=True)
    assert torch.equal(got, want) and torch.equal(top, want_top)
    bias = torch.randn(n, generator=g, device="cuda").to(torch.bfloat16)
    assert torch.equal(linear_nt(x, w, bias, out_dtype=out_dtype), linear_nt(x, w, bias, out_dtype=out_dtype, tile=6))
