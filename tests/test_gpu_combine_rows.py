"""The combine's wave form at the edges of its 512-column pieces, and the widths and alignments it leaves to the other form:
the oracle's bits, with infinities and NaN among the rows."""
import pytest
import torch

from _util import bf16_to_np
from oracle import moe as o_moe
from oracle.prims import bf16_bits

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("tokens", [1, 5, 259])
@pytest.mark.parametrize("width", [8, 120, 128, 152, 160, 248, 256, 504, 512, 520, 2048, 300])
@pytest.mark.parametrize("k", [2, 3, 4, 8])
@pytest.mark.parametrize("offset", [0, 4])
def test_combine_rows(tokens, width, k, offset):
    from isoexec_amd import _lib

    g = torch.Generator().manual_seed(tokens + width + k)
    flat = torch.randn(tokens * k * width + offset, generator=g).to(torch.bfloat16)
    rows = torch.randperm(tokens * k, generator=g).to(torch.int32).view(tokens, k)
    x = flat[offset:].view(tokens * k, width)
    x[0, 0], x[-1, width - 1], x[rows[0, 1].item(), 3], x[rows[0, 0].item(), 3] = (float("nan"), float("inf"),
                                                                                   float("inf"), float("-inf"))
    dev = flat.cuda()
    for fp32 in (0, 1):
        out = torch.empty(tokens, width, dtype=torch.bfloat16, device="cuda")
        rows_d = rows.cuda()
        rc = _lib.lib().ix_moe_combine(dev.data_ptr() + 2 * offset, rows_d.data_ptr(), out.data_ptr(), tokens, width, k, fp32,
                                       _lib.current_stream(dev.device))
        want = bf16_bits(o_moe.combine(bf16_to_np(x), rows.numpy(), fp32_acc=bool(fp32))).view("int16")
        assert rc == 0 and torch.equal(out.view(torch.int16).cpu(), torch.from_numpy(want))
