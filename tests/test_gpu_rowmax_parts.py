"""The row maximum over parts on both sides of the line between its two launches."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("parts", [1, 511, 512, 513, 639, 640, 641, 2376, 5000])
def test_row_maximum_of_parts(parts):
    from isoexec_amd import _lib

    x = torch.randn(37, parts + 3, device="cuda")
    x[3], x[5, parts - 1] = float("-inf"), 9.0
    out = torch.empty(37, device="cuda")
    rc = _lib.lib().ix_rowmax_reduce(x.data_ptr(), parts + 3, parts, 37, out.data_ptr(), _lib.current_stream(x.device))
    assert rc == 0 and torch.equal(out, x[:, :parts].max(dim=1).values)
