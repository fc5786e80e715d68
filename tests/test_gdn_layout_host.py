"""Which layout the delta-rule scan takes by the lengths (``ix_gdn_layout``): a rule of the library, no GPU."""

import pytest

WALK, TWO, ONE = 0, 16, 19


def layout(lens, *, HV=32, V=128, K=128, fp32=False, chunk=0, longest=None):
    from isoexec_amd import _lib

    return _lib.lib().ix_gdn_layout(len(lens), HV, K, V, 0 if fp32 else 1, chunk, sum(lens), max(lens) if longest is None else longest)


def spread(n, lo, hi):
    return [lo + (hi - lo) * i // (n - 1) for i in range(n)]


@pytest.mark.parametrize("lens,plain,boundary", [
    ([8000] + [100] * 15, WALK, WALK), ([4096] + [64] * 31, WALK, WALK), ([8000] + [200] * 47, WALK, WALK),  # one long prompt
    ([8000] + [100] * 63, WALK, WALK), ([4000] * 2 + [200] * 14, WALK, WALK),
    ([2000] * 4 + [200] * 60, ONE, ONE), ([3000] + [500] * 47, ONE, ONE),  # enough beside it for one row per lane, not for two
    ([1000] * 16, ONE, ONE), (spread(16, 60, 1410), ONE, ONE), ([1000] * 48, TWO, ONE), (spread(48, 60, 1470), TWO, ONE),
    ([2560] * 64, TWO, ONE), ([9] * 64, TWO, ONE), ([9] * 48, WALK, ONE), ([1000] * 9, WALK, WALK), ([8192], WALK, WALK)])
def test_the_longest_sequence_decides(lens, plain, boundary):
    assert layout(lens) == plain and layout(lens, chunk=64) == boundary


def test_lengths_that_the_host_does_not_know():
    """Only what no length decides: 2048 workgroups of 128 rows, and never the boundary form."""
    assert layout([1000] * 64, longest=0) == TWO and layout([1000] * 63, longest=0) == WALK
    assert layout([1000] * 200, longest=0, chunk=64) == WALK and layout([1000] * 200, V=64, longest=0) == WALK


def test_what_four_lanes_do_not_serve():
    assert layout([1000] * 64, K=64) == WALK and layout([1000] * 64, V=32) == WALK
    assert layout([1000] * 64, V=64) == ONE  # no groups of 128 rows
    assert layout([1000] * 10, chunk=64) == ONE and layout([1000] * 10, chunk=64, fp32=True) == WALK
    assert layout([], longest=0) == WALK and layout([0] * 64) == TWO
