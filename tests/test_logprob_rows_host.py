"""Which rows the log-softmax keeps on the CU (``ix_logprob_keeps_rows``): a rule of the library, no GPU."""

import pytest

F32, BF16 = 0, 1


def keeps(dtype, rows, V, G):
    from isoexec_amd import _lib

    return bool(_lib.lib().ix_logprob_keeps_rows(dtype, rows, V, G))


@pytest.mark.parametrize("rows,V,G,fp32,bf16", [
    (1000, 151936, 8, True, True), (192, 151936, 8, True, True), (257, 151936, 8, True, True), (191, 151936, 8, False, False),
    (1000, 65528, 8, False, False), (1000, 65536, 8, True, True),
    (256, 65536, 8, True, True), (257, 65536, 8, True, False), (383, 65536, 8, True, False), (257, 73728, 2, True, True),
    (1000, 65536, 64, False, False), (1000, 131072, 64, True, False),                       # blocks a quarter and half full
    (192, 262144, 8, True, False), (384, 262144, 8, True, True), (513, 196608, 32, True, False),  # more than stays in bf16
    (1000, 393216, 8, True, True), (513, 524288, 8, True, False), (1000, 524288, 8, True, True), (1000, 1048576, 8, True, False), (257, 2097152, 8, True, False), (1000, 2097160, 8, False, False)])
def test_rows_are_kept_where_it_measured_faster(rows, V, G, fp32, bf16):
    assert keeps(F32, rows, V, G) == fp32 and keeps(BF16, rows, V, G) == bf16
