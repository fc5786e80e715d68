"""The walk (``k_gdn_walk``: prefill of few sequences, stateless forward, boundary form) at the edges of its tiles."""

import numpy as np
import pytest
import torch

from _util import DevicePrims, bf16_to_np, cpu_gen, np_to_bf16, same_bits
from oracle import gdn as o_gdn

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
EDGES = [17, 1, 0, 16, 33, 15, 48, 2, 31]  # around the tile of 16 tokens (8 for K = 256), an empty sequence


def make(lens, H, HV, K, V, dtype, seed):
    g = cpu_gen(seed)
    T = sum(lens)
    unit = lambda t: t / t.norm(dim=-1, keepdim=True)
    q, k = unit(torch.randn(1, T, H, K, generator=g)), unit(torch.randn(1, T, H, K, generator=g))
    v = torch.randn(1, T, HV, V, generator=g)
    gate = -torch.nn.functional.softplus(torch.randn(1, T, HV, generator=g))
    beta = torch.sigmoid(torch.randn(1, T, HV, generator=g))
    d = lambda t: t.to(dtype).to(DEV)
    return d(q), d(k), d(v), gate.to(DEV), d(beta)


def offsets(lens):
    return torch.tensor([0] + list(np.cumsum(lens)), dtype=torch.int32, device=DEV)


@pytest.mark.parametrize("rows_per_group", [1, 2])
@pytest.mark.parametrize("K,V,dtype", [(32, 128, torch.bfloat16), (64, 64, torch.float32), (64, 64, torch.bfloat16),
                                       (128, 128, torch.bfloat16), (128, 32, torch.float32), (256, 64, torch.bfloat16)])
def test_walk_equals_the_token_staged_scan(K, V, dtype, rows_per_group):
    """Outputs and final states bit for bit against ``k_gdn_scan`` (pinned against the oracle), one and two rows per lane
    group, a null lane and an empty sequence among them; then the stateless forward against the same from zero."""
    from isoexec_amd.ops.gdn.gdn_ops import gdn_recurrent_kernel, stateless_forward

    H, HV = 2, 4
    args = make(EDGES, H, HV, K, V, dtype, K + V)
    cu, N = offsets(EDGES), len(EDGES)
    rows = torch.arange(1, N + 1, dtype=torch.int32, device=DEV)
    rows[4] = 0
    pool0 = torch.randn(N + 1, HV, V, K, generator=cpu_gen(3)).to(DEV)
    run = lambda code, pool, idx: gdn_recurrent_kernel(*args, ssm_state=pool, state_indices=idx, cu_seqlens=cu, time_tile=code)
    pa, pb = pool0.clone(), pool0.clone()
    want = run(16 | (1 << 8), pa, rows)
    got = run((16 + rows_per_group) << 8, pb, rows)
    assert same_bits(got, want) and same_bits(pb, pa)
    rows[4] = 5
    zero = torch.zeros_like(pool0)
    assert same_bits(stateless_forward(*args, cu_seqlens=cu), run(16 | (1 << 8), zero, rows))


@pytest.mark.parametrize("K,H,HV,V,dtype,lens", [
    (32, 2, 4, 64, torch.bfloat16, EDGES), (64, 2, 2, 32, torch.float32, EDGES), (64, 4, 8, 64, torch.bfloat16, [33]),
    (128, 2, 4, 64, torch.bfloat16, EDGES), (128, 1, 1, 16, torch.float32, [1, 50]),  # slices split over two lanes
    (64, 8, 16, 64, torch.bfloat16, EDGES), (64, 8, 32, 64, torch.float32, [16, 8, 1, 40, 17, 3, 5, 2]),  # around its line
    (128, 16, 32, 128, torch.bfloat16, [47]), (128, 16, 32, 128, torch.float32, [32, 17]),  # a staging wave, whole slices
    (128, 16, 32, 128, torch.float32, [47]), (256, 4, 8, 128, torch.float32, [25, 9]),  # in fp32 up to one workgroup per CU
    (256, 4, 8, 128, torch.float32, [25, 9, 16]),
    (128, 8, 16, 128, torch.bfloat16, EDGES), (256, 1, 2, 64, torch.bfloat16, EDGES), (256, 1, 2, 64, torch.float32, [9])])
def test_walk_by_the_rule_equals_the_token_staged_scan(K, H, HV, V, dtype, lens):
    """The forms that the number of workgroups chooses (a staging wave, split slices, neither): output and final state bit for
    bit against ``k_gdn_scan``, with and without a state."""
    from isoexec_amd.ops.gdn.gdn_ops import gdn_recurrent_kernel, stateless_forward

    args = make(lens, H, HV, K, V, dtype, K + V + HV)
    cu, N = offsets(lens), len(lens)
    rows = torch.arange(1, N + 1, dtype=torch.int32, device=DEV)
    pa = torch.randn(N + 1, HV, V, K, generator=cpu_gen(4)).to(DEV)
    pb, zero = pa.clone(), torch.zeros_like(pa)
    run = lambda code, pool: gdn_recurrent_kernel(*args, ssm_state=pool, state_indices=rows, cu_seqlens=cu, time_tile=code)
    want = run(16 | (1 << 8), pa)
    assert same_bits(run(0, pb), want) and same_bits(pb, pa)
    assert same_bits(stateless_forward(*args, cu_seqlens=cu), run(16 | (1 << 8), zero))


@pytest.mark.parametrize("K,H,HV,V,dtype,n", [
    (64, 2, 4, 64, torch.bfloat16, 3), (128, 2, 4, 64, torch.float32, 3),  # slices split over two lanes
    (128, 16, 32, 128, torch.bfloat16, 2), (64, 16, 32, 64, torch.float32, 8), (256, 2, 4, 64, torch.bfloat16, 3),  # whole slices
    (128, 16, 32, 128, torch.float32, 1)])
def test_null_lane_beside_a_staging_wave(K, H, HV, V, dtype, n):
    """Sequences without a state row: outputs zero, the pool's other rows as in ``k_gdn_scan``, the null row untouched."""
    from isoexec_amd.ops.gdn.gdn_ops import gdn_recurrent_kernel

    lens = [33, 16, 5, 18, 1, 40, 31, 2][:n]
    args = make(lens, H, HV, K, V, dtype, n)
    cu = offsets(lens)
    rows = torch.arange(1, n + 1, dtype=torch.int32, device=DEV)
    rows[n // 2] = 0
    pa = torch.randn(n + 1, HV, V, K, generator=cpu_gen(6)).to(DEV)
    pb = pa.clone()
    run = lambda code, pool: gdn_recurrent_kernel(*args, ssm_state=pool, state_indices=rows, cu_seqlens=cu, time_tile=code)
    want, got = run(16 | (1 << 8), pa), run(0, pb)
    assert same_bits(got, want) and same_bits(pb, pa)
    a, b = sum(lens[:n // 2]), sum(lens[:n // 2 + 1])
    assert not got[0, a:b].any() and (n == 1 or got.any())


def test_more_sequences_than_a_workgroup_ranks():
    from isoexec_amd.ops.gdn.gdn_ops import gdn_recurrent_kernel, stateless_forward

    lens = [(7 * i) % 23 for i in range(260)]
    args = make(lens, 1, 2, 64, 64, torch.bfloat16, 5)
    cu = offsets(lens)
    rows = torch.arange(1, len(lens) + 1, dtype=torch.int32, device=DEV)
    pool = torch.zeros(len(lens) + 1, 2, 64, 64, device=DEV)
    want = gdn_recurrent_kernel(*args, ssm_state=pool, state_indices=rows, cu_seqlens=cu, time_tile=16 | (1 << 8))
    assert same_bits(stateless_forward(*args, cu_seqlens=cu), want)


@pytest.mark.parametrize("chunk", [16, 48, 64])
@pytest.mark.parametrize("K,H,HV", [(64, 2, 4), (128, 1, 2), (256, 1, 1)])
def test_boundary_form_in_one_walk_against_the_oracle(K, H, HV, chunk):
    from isoexec_amd.ops.gdn.gdn_cpr import gdn_cpr_fwd

    lens = [chunk, 1, 2 * chunk + 5, 0, 130, chunk + 16, 15]
    q, k, v, gate, beta = make(lens, H, HV, K, 64, torch.bfloat16, chunk)
    f = lambda t: bf16_to_np(t[0].cpu())
    want, _, _ = o_gdn.cpr_forward(f(q), f(k), f(v), gate[0].cpu().numpy(), f(beta), lens, chunk, prims=DevicePrims(DEV))
    assert same_bits(gdn_cpr_fwd(q, k, v, gate, beta, cu_seqlens=offsets(lens), chunk_size=chunk)[0].cpu(), np_to_bf16(want))


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("K,V,n", [(128, 128, 1), (128, 128, 2), (128, 128, 4), (128, 128, 9), (64, 64, 5), (64, 64, 8), (64, 64, 16),
                                   (64, 64, 33), (256, 64, 2), (256, 64, 4), (256, 64, 17)])
def test_boundary_form_by_the_rule_equals_few_heads_alone(K, V, n, dtype):
    """Whole slices with a staging wave, without one, and two rows a lane group, as 32 heads and n sequences choose them, against
    the same sequence and four heads of it in a call of their own (split slices up to K = 128, which the oracle test above
    covers; whole slices with a staging wave at K = 256): at least three chunks, lengths around the tile and the chunk."""
    from isoexec_amd.ops.gdn.gdn_ops import stateless_forward

    H, HV, chunk = 16, 32, 32
    lens = [(2 * chunk + 13 * i * i) % 101 + 1 for i in range(n)]
    q, k, v, gate, beta = args = make(lens, H, HV, K, V, dtype, K + n)
    got = stateless_forward(*args, cu_seqlens=offsets(lens), chunk_size=chunk)
    at = 0
    for i, length in enumerate(lens):
        t, h = slice(at, at + length), 2 * (i % 8)
        at += length
        alone = stateless_forward(q[:, t, h:h + 2].contiguous(), k[:, t, h:h + 2].contiguous(), v[:, t, 2 * h:2 * h + 4].contiguous(),
                                  gate[:, t, 2 * h:2 * h + 4].contiguous(), beta[:, t, 2 * h:2 * h + 4].contiguous(),
                                  cu_seqlens=offsets([length]), chunk_size=chunk)
        assert same_bits(got[:, t, 2 * h:2 * h + 4], alone), (i, length)


def test_lane_pairs_of_many_sequences_with_the_norm_folded_in():
    """2048 (sequence, head) pairs: the lane-pair layout, longest sequence first, with and without a state pool, and with the
    gated output norm in its launch; against the walk followed by the norm."""
    from isoexec_amd.ops.gdn.gdn_ops import gdn_recurrent_kernel, stateless_forward
    from isoexec_amd.ops.norms.fused_outnorm import fused_gated_out_norm

    H, HV, K, V = 16, 32, 128, 128
    lens = [(11 * i) % 19 for i in range(64)]
    T, N = sum(lens), len(lens)
    args = make(lens, H, HV, K, V, torch.bfloat16, 8)
    cu = offsets(lens)
    z = torch.randn(T, HV, V, generator=cpu_gen(1)).to(torch.bfloat16).to(DEV)
    w = (0.1 * torch.randn(V, generator=cpu_gen(2))).to(torch.bfloat16).to(DEV)
    rows = torch.arange(1, N + 1, dtype=torch.int32, device=DEV)
    pa = torch.zeros(N + 1, HV, V, K, device=DEV)
    pb = pa.clone()
    want = gdn_recurrent_kernel(*args, ssm_state=pa, state_indices=rows, cu_seqlens=cu, time_tile=17 << 8)
    normed = fused_gated_out_norm(want[0], z, w, 1e-6).view(1, T, HV, V)
    assert same_bits(stateless_forward(*args, cu_seqlens=cu), want)
    assert same_bits(stateless_forward(*args, cu_seqlens=cu, gated_norm=(z, w, 1e-6, True)), normed)
    got = gdn_recurrent_kernel(*args, ssm_state=pb, state_indices=rows, cu_seqlens=cu, gated_norm=(z, w, 1e-6, True))
    assert same_bits(got, normed) and same_bits(pb, pa)
