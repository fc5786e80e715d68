"""The log-softmax's row kept on the CU (``k_lp_row_held``) against the same rows read twice and split over workgroups."""

import pytest
import torch

from _util import cpu_gen, same_bits

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


# Columns: the line, blocks that a wave keeps in registers, in LDS and reads again, a leaf that ends with eight columns of a
# block, one leaf, 64 leaves, more blocks than are kept. Rows: the fewest of this shape, a workgroup with two, and with a third.
@pytest.mark.parametrize("V,G", [(65536, 8), (65600, 1), (8 * 12296, 8), (151936, 8), (64 * 4104, 64), (262144, 4), (81920, 2)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("rows", [192, 257, 514])
def test_kept_rows_equal_the_other_shapes(V, G, dtype, rows):
    from isoexec_amd.ops.logprobs.rowinv import sampled_forward

    g = cpu_gen(V + rows)
    base = 3.0 * torch.randn(1, V + 8 * rows, generator=g)
    x = base.as_strided((rows, V), (8, 1)).to(dtype).to(DEV)  # rows shifted by eight columns each
    inf = float("inf")
    x[3] = -inf
    x[4, 17] = inf
    x[5, V - 1] = float("nan")
    x[6, : V // 2] = -inf
    x[rows - 1, V - 1] = 50.0
    t = torch.randint(0, V, (rows,), generator=g).to(DEV)
    t[1], t[2] = -100, V
    got = sampled_forward(x, t, G)
    for shape in (1, 2):
        want = sampled_forward(x, t, G, force_shape=shape)
        assert same_bits(torch.nan_to_num(got[0], 7e7), torch.nan_to_num(want[0], 7e7)), shape
        assert same_bits(torch.nan_to_num(got[1], 7e7), torch.nan_to_num(want[1], 7e7)), shape


def test_kept_rows_with_a_longer_row_stride():
    from isoexec_amd.ops.logprobs.rowinv import sampled_forward

    wide = torch.randn(300, 65536 + 64, generator=cpu_gen(1)).to(DEV)
    x, t = wide[:, 32:32 + 65536], torch.randint(0, 65536, (300,), generator=cpu_gen(2)).to(DEV)
    got, want = sampled_forward(x, t, 8), sampled_forward(x.contiguous(), t, 8, force_shape=2)
    assert same_bits(got[0], want[0]) and same_bits(got[1], want[1])
