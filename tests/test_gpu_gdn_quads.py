"""The four-lane layouts of the delta-rule scan (K = 128): the state's update on the matrix pipe against the multiply-adds of
the token-staged scan (``k_gdn_scan``, pinned against the oracle)."""

import pytest
import torch

from _util import cpu_gen, same_bits

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
LENS = [1, 3, 4, 5, 15, 16, 17, 0, 33]  # around four tokens of a loop step and the tile of 16; an empty sequence


def operands(lens, H, HV, V, dtype, seed):
    g = cpu_gen(seed)
    T = sum(lens)
    unit = lambda t: t / t.norm(dim=-1, keepdim=True)
    q, k = unit(torch.randn(1, T, H, 128, generator=g)), unit(torch.randn(1, T, H, 128, generator=g))
    v = torch.randn(1, T, HV, V, generator=g)
    gate = -torch.nn.functional.softplus(torch.randn(1, T, HV, generator=g))
    beta = torch.sigmoid(torch.randn(1, T, HV, generator=g))
    cu = torch.tensor([0] + list(torch.tensor(lens).cumsum(0)), dtype=torch.int32, device=DEV)
    d = lambda t: t.to(dtype).to(DEV)
    return (d(q), d(k), d(v), gate.to(DEV), d(beta)), cu


# A product of one term per element rounds once, like fmaf, whatever the size of the operands: a state of ordinary size, one
# that is subnormal with updates that are subnormal too, and one near the largest value.
@pytest.mark.parametrize("size", [1.0, 3e-39, 1e38])
@pytest.mark.parametrize("V,dtype", [(128, torch.bfloat16), (256, torch.float32)])
def test_update_on_the_matrix_pipe_rounds_as_the_multiply_adds(V, dtype, size):
    from isoexec_amd.ops.gdn.gdn_ops import gdn_recurrent_kernel

    H, HV, N = 2, 4, len(LENS)
    args, cu = operands(LENS, H, HV, V, dtype, V)
    if size < 1.0:
        args = args[:2] + (args[2] * 1e-38,) + args[3:]
    start = (size * torch.randn(N + 1, HV, V, 128, generator=cpu_gen(3))).to(DEV)
    rows = torch.tensor([1, 2, 3, 0, 5, 6, 7, 8, 9], dtype=torch.int32, device=DEV)  # the fourth is a null lane
    pa, pb = start.clone(), start.clone()
    want = gdn_recurrent_kernel(*args, ssm_state=pa, state_indices=rows, cu_seqlens=cu, time_tile=16 | (1 << 8))
    got = gdn_recurrent_kernel(*args, ssm_state=pb, state_indices=rows, cu_seqlens=cu, time_tile=16 << 8)
    assert same_bits(got, want) and same_bits(pb, pa)
    assert not same_bits(pa, start)


@pytest.mark.parametrize("V,dtype", [(128, torch.bfloat16), (64, torch.float32)])
def test_walk_with_four_lanes_per_row_equals_the_token_staged_scan(V, dtype):
    """Code 19: outputs, final states and a null lane, one row block and two."""
    from isoexec_amd.ops.gdn.gdn_ops import gdn_recurrent_kernel

    H, HV, N = 2, 4, len(LENS)
    args, cu = operands(LENS, H, HV, V, dtype, V)
    pa = torch.randn(N + 1, HV, V, 128, generator=cpu_gen(3)).to(DEV)
    pb = pa.clone()
    rows = torch.tensor([1, 2, 3, 0, 5, 6, 7, 8, 9], dtype=torch.int32, device=DEV)
    run = lambda code, pool: gdn_recurrent_kernel(*args, ssm_state=pool, state_indices=rows, cu_seqlens=cu, time_tile=code)
    assert same_bits(run(19 << 8, pb), run(16 | (1 << 8), pa)) and same_bits(pb, pa)


# Enough workgroups for four lanes per row, by the rule: 132 sequences (the last turn through the CUs is not a whole one) of the
# lengths above, plain and in the boundary form, against the same sequences nine at a time (the sixteen-lane walk).
@pytest.mark.parametrize("HV,dtype", [(8, torch.bfloat16), (16, torch.float32)])
@pytest.mark.parametrize("chunk", [0, 16, 32])
def test_walk_with_four_lanes_per_row_by_the_rule(HV, dtype, chunk):
    from isoexec_amd.ops.gdn.gdn_ops import stateless_forward

    lens = [LENS[i % 9] + (i // 9) % 2 for i in range(132)]  # one row block per head: 132 * HV workgroups
    args, cu = operands(lens, HV // 2, HV, 64, dtype, HV + chunk)
    got = stateless_forward(*args, cu_seqlens=cu, chunk_size=chunk)
    at = 0
    for i in range(0, len(lens), 9):
        part = lens[i:i + 9]
        t = slice(at, at + sum(part))
        at += sum(part)
        _, few = operands(part, 1, 1, 1, dtype, 0)
        alone = stateless_forward(*(a[:, t].contiguous() for a in args), cu_seqlens=few, chunk_size=chunk)
        assert same_bits(got[:, t], alone), i
