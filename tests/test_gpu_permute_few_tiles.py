"""The permutation at the edges of the launch that does prefix, offsets and scatter at once (2 .. 64 token tiles): against a
stable sort on the host, with expert counts that do not divide the workgroup, experts without rows and a ragged last tile."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("t", [257, 512, 700, 48 * 256, 48 * 256 + 1, 64 * 256, 64 * 256 + 1])
@pytest.mark.parametrize("e,k", [(128, 8), (3, 2), (60, 4), (512, 16)])
def test_permutation(t, e, k):
    from isoexec_amd.ops.moe.moe_hip import permute

    g = torch.Generator().manual_seed(t + e)
    used = max(k, e - 2)  # the last two experts get nothing where there are enough
    idx = torch.rand(t, used, generator=g).topk(k, dim=1).indices.to(torch.int32)
    prob = torch.rand(t, k, generator=g)
    p = permute(idx.cuda(), prob.cuda(), e, BM=96)
    flat = idx.reshape(-1).long()
    order = torch.sort(flat * t + torch.arange(t).repeat_interleave(k)).indices  # expert-major, token-ascending
    counts = torch.bincount(flat, minlength=e)
    starts = torch.cat([torch.zeros(1, dtype=torch.long), counts.cumsum(0)])
    assert torch.equal(p.counts.cpu().long(), counts) and torch.equal(p.offsets.cpu().long(), starts)
    assert torch.equal(p.sorted_token.cpu().long(), order // k)
    assert torch.equal(p.permuted_prob.cpu(), prob.reshape(-1)[order])
    pos = torch.empty(t * k, dtype=torch.long)
    pos[order] = torch.arange(t * k)
    assert torch.equal(p.combine_rows.cpu().long(), pos.view(t, k).sort(dim=1).values)
    meta, n = p.tile_meta.cpu(), p.max_tiles
    want = [(x, int(starts[x]) + r, min(96, int(counts[x]) - r)) for x in range(e) for r in range(0, int(counts[x]), 96)]
    assert int(meta[0]) == len(want)
    got = meta[1:].view(3, n)[:, : len(want)].t().tolist()
    assert [tuple(v) for v in got] == want
