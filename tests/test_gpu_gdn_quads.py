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


def nan_alike(a, b):
    """Equal bits, but for a NaN's: which of two NaN operands an instruction passes on is not part of the contract."""
    n = lambda t: torch.where(t.isnan(), torch.full_like(t, 7e7), t)
    return same_bits(n(a), n(b))


# Signed zeros, infinities and NaNs in the state and in the values, keys and queries of zero, on both four-lane layouts against the
# sixteen-lane scan. The first sequence has one token: its infinity is still one in the state.
@pytest.mark.parametrize("code", [16, 19])
@pytest.mark.parametrize("V,dtype", [(128, torch.bfloat16), (128, torch.float32)])
def test_special_values_on_four_lanes_per_row(V, dtype, code):
    from isoexec_amd.ops.gdn.gdn_ops import gdn_recurrent_kernel

    H, HV, N = 2, 4, len(LENS)
    (q, k, v, gate, beta), cu = operands(LENS, H, HV, V, dtype, code)
    start = torch.randn(N + 1, HV, V, 128, generator=cpu_gen(3)).to(DEV)
    start[1] = 0.0
    start[2] = -0.0
    start[3, :, ::3] = -0.0
    start[5, 0, 5, 7], start[5, 1, 6, 100] = float("inf"), -float("inf")
    start[6, 2, 9, 64] = float("nan")
    start[7, :, :, 1::2] = 0.0
    v, k, q = v.clone(), k.clone(), q.clone()
    v[0, ::4] = -0.0
    v[0, 0, 0, 9], v[0, 40, 1, 3], v[0, 41, 2, 4], v[0, 60, 3, 5] = float("inf"), float("inf"), -float("inf"), float("nan")
    k[0, 5], q[0, 6] = 0.0, -0.0
    rows = torch.tensor([1, 2, 3, 0, 5, 6, 7, 8, 9], dtype=torch.int32, device=DEV)
    pa, pb = start.clone(), start.clone()
    run = lambda c, pool: gdn_recurrent_kernel(q, k, v, gate, beta, ssm_state=pool, state_indices=rows, cu_seqlens=cu, time_tile=c)
    want, got = run(16 | (1 << 8), pa), run(code << 8, pb)
    assert nan_alike(got.float(), want.float()) and nan_alike(pb, pa)
    assert int(want.isnan().sum()) > 0 and int(pa[1].isinf().sum()) > 0 and int(pa[9].isnan().sum()) == 0


# The state returns exactly the value that arrives: the update is a product with zero, of either sign.
@pytest.mark.parametrize("code", [16, 19])
def test_a_state_that_returns_the_value_exactly(code):
    from isoexec_amd.ops.gdn.gdn_ops import gdn_recurrent_kernel

    HV, V, T = 4, 128, 6
    k = torch.zeros(1, T, HV, 128, device=DEV)
    k[..., 5] = 1.0
    pool = torch.randn(2, HV, V, 128, generator=cpu_gen(1)).to(DEV)
    v = pool[1, :, :, 5].expand(1, T, HV, V).contiguous()
    gate, beta = torch.zeros(1, T, HV, device=DEV), torch.full((1, T, HV), 0.5, device=DEV)
    q = torch.randn(1, T, HV, 128, generator=cpu_gen(2)).to(DEV)
    cu, rows = torch.tensor([0, T], dtype=torch.int32, device=DEV), torch.tensor([1], dtype=torch.int32, device=DEV)
    start = pool.clone()
    got = gdn_recurrent_kernel(q, k, v, gate, beta, ssm_state=pool, state_indices=rows, cu_seqlens=cu, time_tile=code << 8)
    other = start.clone()
    want = gdn_recurrent_kernel(q, k, v, gate, beta, ssm_state=other, state_indices=rows, cu_seqlens=cu, time_tile=16 | (1 << 8))
    assert same_bits(pool, start) and same_bits(got, want)


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


# By the rule: 132 sequences (the last turn through the CUs is not a whole one) and 300 (more than are ranked by length), plain and
# in the boundary form, against the same sequences nine at a time (the sixteen-lane walk). q, k and v are column blocks of one
# buffer with columns of its own, as a layer's convolution leaves them.
@pytest.mark.parametrize("n,HV,dtype", [(132, 16, torch.bfloat16), (132, 16, torch.float32), (300, 8, torch.bfloat16)])
@pytest.mark.parametrize("chunk", [0, 16, 32])
def test_walk_with_four_lanes_per_row_by_the_rule(n, HV, dtype, chunk):
    from isoexec_amd import _lib
    from isoexec_amd.ops.gdn.gdn_ops import stateless_forward

    H, V = HV // 2, 64
    lens = [LENS[i % 9] and LENS[i % 9] + 20 + (i // 9) % 2 for i in range(n)]
    T = sum(lens)
    assert _lib.lib().ix_gdn_layout(n, HV, 128, V, _lib.dtype_code(dtype), chunk, T, max(lens)) == 19
    (q, k, v, gate, beta), cu = operands(lens, H, HV, V, dtype, HV + chunk)
    wide = torch.zeros(1, T, 2 * H * 128 + HV * V + 8, dtype=dtype, device=DEV)
    parts = wide[..., :H * 128], wide[..., H * 128:2 * H * 128], wide[..., 2 * H * 128:2 * H * 128 + HV * V]
    args = [p.unflatten(2, t.shape[2:]) for p, t in zip(parts, (q, k, v))]
    for p, t in zip(args, (q, k, v)):
        p.copy_(t)
    got = stateless_forward(*args, gate, beta, cu_seqlens=cu, chunk_size=chunk, longest=max(lens))
    at = 0
    for i in range(0, n, 9):
        part = lens[i:i + 9]
        t = slice(at, at + sum(part))
        at += sum(part)
        _, few = operands(part, 1, 1, 1, dtype, 0)
        alone = stateless_forward(*(a[:, t].contiguous() for a in (q, k, v, gate, beta)), cu_seqlens=few, chunk_size=chunk)
        assert same_bits(got[:, t], alone), i


# One long sequence and many short ones, an even spread and equal lengths: the three layouts, with a state pool and without, with the
# gated norm and without. The form whose lengths the host does not know takes another layout for the same sequences.
@pytest.mark.parametrize("lens,layout", [([300] + [3] * 15, 0), ([80 - 2 * i for i in range(16)], 19), ([24] * 48, 16),
                                         ([300] + [3] * 63, 0), ([5] * 64, 16)])
def test_lengths_known_on_the_host_change_no_bits(lens, layout):
    from isoexec_amd import _lib
    from isoexec_amd.ops.gdn.gdn_ops import gdn_recurrent_kernel, stateless_forward
    from isoexec_amd.ops.norms.fused_outnorm import fused_gated_out_norm

    H, HV, V, N, T = 16, 32, 128, len(lens), sum(lens)
    assert _lib.lib().ix_gdn_layout(N, HV, 128, V, 1, 0, T, max(lens)) == layout
    args, cu = operands(lens, H, HV, V, torch.bfloat16, N)
    rows = torch.arange(1, N + 1, dtype=torch.int32, device=DEV)
    z = torch.randn(T, HV, V, generator=cpu_gen(1)).to(torch.bfloat16).to(DEV)
    w = (0.1 * torch.randn(V, generator=cpu_gen(2))).to(torch.bfloat16).to(DEV)
    norm = (z, w, 1e-6, True)
    start = torch.randn(N + 1, HV, V, 128, generator=cpu_gen(3)).to(DEV)
    run = lambda pool, **kw: gdn_recurrent_kernel(*args, ssm_state=pool, state_indices=rows, cu_seqlens=cu, **kw)
    pools = [start.clone() for _ in range(3)]
    want = run(pools[0], time_tile=16 | (1 << 8))
    normed = fused_gated_out_norm(want[0], z, w, 1e-6).view(1, T, HV, V)
    assert same_bits(run(pools[1], longest=max(lens)), want) and same_bits(pools[1], pools[0])
    assert same_bits(run(pools[2], longest=max(lens), gated_norm=norm), normed) and same_bits(pools[2], pools[0])
    zero = torch.zeros_like(start)
    want = run(zero, time_tile=16 | (1 << 8))
    normed = fused_gated_out_norm(want[0], z, w, 1e-6).view(1, T, HV, V)
    assert same_bits(stateless_forward(*args, cu_seqlens=cu, longest=max(lens)), want)
    assert same_bits(stateless_forward(*args, cu_seqlens=cu, longest=max(lens), gated_norm=norm), normed)
