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
    got = sampled_forward(x, t, G, force_shape=3)
    for shape in (0, 1, 2):
        want = sampled_forward(x, t, G, force_shape=shape)
        assert same_bits(torch.nan_to_num(got[0], 7e7), torch.nan_to_num(want[0], 7e7)), shape
        assert same_bits(torch.nan_to_num(got[1], 7e7), torch.nan_to_num(want[1], 7e7)), shape


def test_kept_rows_with_a_longer_row_stride():
    from isoexec_amd.ops.logprobs.rowinv import sampled_forward

    wide = torch.randn(300, 65536 + 64, generator=cpu_gen(1)).to(DEV)
    x, t = wide[:, 32:32 + 65536], torch.randint(0, 65536, (300,), generator=cpu_gen(2)).to(DEV)
    got, want = sampled_forward(x, t, 8, force_shape=3), sampled_forward(x.contiguous(), t, 8, force_shape=2)
    assert same_bits(got[0], want[0]) and same_bits(got[1], want[1])


# Segments of 8192 columns that end with a group of eight, one row and several, a row that no 16-byte store fits, a maximum that is
# given; the row's log-sum joined by every segment for itself, and by a launch in front (a leaf of more than 256 blocks).
@pytest.mark.parametrize("V,G,pad", [(8, 1, 0), (8192, 8, 0), (8200, 1, 0), (151936, 8, 0), (151936, 8, 1), (1000, 8, 0), (16392, 1, 4),
                                     (256 * 4096, 1, 0), (256 * 4096 + 8, 1, 4), (2 * 257 * 4096, 2, 1)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_full_rows_of_the_split_shape(V, G, pad, dtype):
    from isoexec_amd import _lib
    from isoexec_amd.ops.logprobs.rowinv import full_forward, sampled_forward

    rows = 5
    g = cpu_gen(V + pad)
    x = (4.0 * torch.randn(rows, V, generator=g)).to(dtype).to(DEV)
    x[1] = -float("inf")
    x[2, V // 2] = float("inf")
    x[3, 0] = float("nan")
    t = torch.full((rows,), V - 1, device=DEV)
    lp, lse = sampled_forward(x, t, G, force_shape=1)
    top = x.float().amax(dim=1) if not pad else None
    if top is not None:
        top[3] = sampled_max(x[3])
    for row_max in (None, top):
        out, got_lse = torch.full((rows, V + pad), 7.0, device=DEV), torch.empty(rows, device=DEV)
        ws = torch.empty(int(_lib.lib().ix_logprob_workspace_bytes(rows, V, G)), dtype=torch.uint8, device=DEV)
        rc = _lib.lib().ix_logprob_rowinv_full(x.data_ptr(), _lib.dtype_code(dtype), rows, V, V, G, out.data_ptr(), V + pad,
                                               got_lse.data_ptr(), ws.data_ptr(), ws.numel(), 2, _lib.ptr(row_max),
                                               _lib.current_stream(x.device))
        assert rc == _lib.IX_OK
        n = lambda a: torch.nan_to_num(a, 7e7)
        assert same_bits(n(got_lse), n(lse)) and same_bits(n(out[:, V - 1]), n(lp)) and (out[:, V:] == 7.0).all()
        want = torch.empty(rows, V, device=DEV)
        rc = _lib.lib().ix_logprob_rowinv_full(x.data_ptr(), _lib.dtype_code(dtype), rows, V, V, G, want.data_ptr(), V, None,
                                               ws.data_ptr(), ws.numel(), 1, None, _lib.current_stream(x.device))
        assert rc == _lib.IX_OK and same_bits(n(out[:, :V]), n(want))
    if G == 8 and not pad:
        assert same_bits(n(full_forward(x, G)), n(want))


def sampled_max(row):
    """The maximum as the kernels take it: a NaN does not count."""
    return row.float()[~row.isnan()].max()
