"""Expert tiles whose height the counts decide on the device (160 or 192, or 256 rows), and bands with several tiles per workgroup: the
maps against those of one height, the products bit for bit against 32-row tiles."""
import math

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(seed)


def _routing(t, e, k, hot, seed):
    """Even routing, or `hot` experts in every token's choice."""
    g = _gen(seed)
    score = torch.rand(t, e, generator=g, device=DEV)
    score[:, torch.randperm(e, generator=g, device=DEV)[:hot]] += 2.0
    return score.topk(k, dim=1).indices.to(torch.int32), torch.rand(t, k, generator=g, device=DEV)


def _height(counts, low_rows, hd, f):
    def cost(rows, us):
        tiles = sum(-(-c // rows) for c in counts)
        turns = lambda x: math.floor(x) + (0.68 + 0.32 * (x % 1.0) if x % 1.0 else 0.0)
        return us * (turns(tiles * (f // 128) / 256) * (hd // 64) + turns(tiles * (hd // 256) / 256) * (f // 64))

    low, tall = cost(low_rows, {160: 1.27, 192: 1.41}[low_rows]), cost(256, 1.64)
    assert abs(tall - low) > 1e-4 * low or not low  # not a case that fp32 decides
    return 256 if tall <= low else low_rows


def _tiles(meta, n):
    return int(meta[0]), meta[1:].view(3, n)[:, : int(meta[0])].cpu()


# even routing takes 160 where two tiles hold what three of 256 would waste, popular experts leave the others one tile of 160
@pytest.mark.parametrize("t,e,k,hot", [
    (3840, 128, 8, 0), (4480, 128, 8, 0), (4480, 128, 8, 4), (4096, 128, 8, 4), (6300, 128, 8, 0), (2900, 96, 8, 3), (300, 3, 3, 0),
    (12289, 512, 8, 0), (16640, 130, 2, 1), (17000, 512, 8, 4)])  # the last three: more counts than one launch takes
@pytest.mark.parametrize("low_rows", [160, 192])
def test_map_by_counts(t, e, k, hot, low_rows):
    from isoexec_amd.ops.moe.moe_hip import permute

    idx, prob = _routing(t, e, k, hot, t + e)
    hd, f = 2048, 768
    p = permute(idx, prob, e, BM=low_rows, layer=(hd, f))
    want_rows = _height(p.counts.tolist(), low_rows, hd, f)
    want = permute(idx, prob, e, BM=want_rows)
    for name in ("counts", "offsets", "sorted_token", "permuted_prob", "combine_rows"):
        assert torch.equal(getattr(p, name), getattr(want, name)), name
    low, tall = (p.tile_meta, p.max_tiles), p.tall
    chosen, other = (tall, low) if want_rows == 256 else (low, tall)
    n, tiles = _tiles(*chosen)
    want_n, want_tiles = _tiles(want.tile_meta, want.max_tiles)
    assert n == want_n and torch.equal(tiles, want_tiles) and int(other[0][0]) == 0


def test_both_heights_are_chosen():
    assert _height([240] * 128, 160, 2048, 768) == 256 and _height([280] * 128, 160, 2048, 768) == 160
    assert _height([240] * 128, 192, 2048, 768) == 256 and _height([330] * 128, 192, 2048, 768) == 192


@pytest.mark.parametrize("dtype", [torch.int32, torch.int64])
@pytest.mark.parametrize("counts", [[280] * 128, [240] * 128, [300, 0] * 64, [132] * 124 + [4000] * 4, [2 ** 31 - 1] * 128, [0] * 128])
@pytest.mark.parametrize("low_rows", [160, 192])
def test_block_map_by_counts(counts, dtype, low_rows):
    from isoexec_amd import _lib

    L = _lib.lib()
    e, hd, f, rows = len(counts), 2048, 768, min(sum(counts), 36000)
    kept = []
    for c in counts:
        kept.append(min(c, rows - sum(kept)))
    c = torch.tensor(counts, dtype=dtype, device=DEV)
    maps = []
    for bm in (low_rows, 256):
        n = int(L.ix_moe_max_tiles(rows, 1, e, bm))
        maps.append((bm, torch.full((1 + 3 * n,), -7, dtype=torch.int32, device=DEV), n))
    (_, m0, n0), (_, m1, n1) = maps
    off = torch.empty(e + 1, dtype=torch.int32, device=DEV)
    stream = _lib.current_stream(torch.device(DEV))
    assert L.ix_moe_block_map_by_counts(c.data_ptr(), int(dtype is torch.int64), e, low_rows, hd, f, rows, off.data_ptr(), m0.data_ptr(),
                                        n0, m1.data_ptr(), n1, stream) == 0
    starts = [0]
    for x in kept:
        starts.append(starts[-1] + x)
    assert off.tolist() == starts
    height = _height(kept, low_rows, hd, f)
    for bm, meta, n in maps:
        got_n, got = _tiles(meta, n)
        want = [(i, starts[i] + r, min(bm, kept[i] - r)) for i in range(e) for r in range(0, kept[i], bm)] if bm == height else []
        assert got_n == len(want) and [tuple(v) for v in got.t().tolist()] == want


def _layer(e, hd, f, seed):
    g = _gen(seed)
    w = lambda *shape: (torch.randn(*shape, generator=g, device=DEV) * 0.03).to(torch.bfloat16)
    return w(e, 2 * f, hd), w(e, hd, f)


@pytest.mark.parametrize("bm,t,hot", [(96, 800, 0), (96, 800, 3), (160, 1500, 0), (160, 2900, 3), (192, 1700, 0), (192, 2900, 3)])
@pytest.mark.parametrize("hd,f", [(1024, 768), (1280, 896)])
def test_bands_of_several_tiles_per_workgroup(bm, t, hot, hd, f):
    """At least two tiles of either product for every workgroup: the next tile's rows are gathered and the chain of the tile
    before runs under a tile's own matrix instructions."""
    from isoexec_amd.ops.moe.moe_hip import experts_forward, permute

    e, k = 128, 8
    w1, w2 = _layer(e, hd, f, 11)
    idx, prob = _routing(t, e, k, hot, t)
    x = torch.randn(t, hd, generator=_gen(t), device=DEV).to(torch.bfloat16)
    p = permute(idx, prob, e, BM=bm)
    assert int(p.tile_meta[0]) * min(f // 128, hd // 256) >= 2 * 256
    got, gi = experts_forward(x, w1, w2, p, return_inter=True)
    want, wi = experts_forward(x, w1, w2, permute(idx, prob, e, BM=32), return_inter=True)
    assert torch.equal(gi, wi) and torch.equal(got, want)


def test_layer_by_counts_eager_and_captured():
    """The layer with even and with popular experts, each height chosen by one of them: eager, and replayed from one graph whose
    routing changes between the replays."""
    from isoexec_amd import _lib
    from isoexec_amd.ops.moe.moe_hip import moe_ffn_forward, route_and_permute
    from isoexec_amd.ops.mm.mm_hip import router_gemm

    t, e, k, hd, f = 4480, 128, 8, 1024, 768
    assert _lib.lib().ix_moe_pick_low_bm(t, k, e, hd, f) == 160
    w1, w2 = _layer(e, hd, f, 12)
    router = (torch.randn(e, hd, generator=_gen(1), device=DEV) * 0.02).to(torch.bfloat16)
    x = torch.randn(t, hd, generator=_gen(2), device=DEV).to(torch.bfloat16)
    biases = [torch.zeros(e, device=DEV), torch.zeros(e, device=DEV)]
    biases[1][:2] = 30.0
    run = lambda bias, **kw: moe_ffn_forward(x, router, w1, w2, k, pre_softmax=True, logit_bias=bias, **kw)
    want = [run(b, BM=32) for b in biases]
    for b, w, tall in zip(biases, want, (False, True)):
        p = route_and_permute(router_gemm(x, router) + b, k, pre_softmax=True, BM=160, layer=(hd, f))[2]
        assert (int(p.tall[0][0]) > 0, int(p.tile_meta[0]) > 0) == (tall, not tall)
        assert torch.equal(run(b), w)
    static = biases[0].clone()
    stream = torch.cuda.Stream()
    stream.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(stream):
        run(static)
    torch.cuda.current_stream().wait_stream(stream)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = run(static)
    for i in (0, 1, 1, 0, 1):
        static.copy_(biases[i])
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, want[i]), i
        assert torch.equal(run(static), want[i])


@pytest.mark.parametrize("hot", [0, 2])
def test_grouped_rows_by_counts(hot):
    """``SequentialMLP.forward``'s door at a size where the counts decide, against the layer's own experts."""
    from types import SimpleNamespace

    from isoexec_amd import _lib
    from isoexec_amd.ops.moe import moe_doors
    from isoexec_amd.ops.moe.moe_hip import experts_forward, permute

    t, e, k, hd, f = 4480, 128, 8, 1024, 768
    assert _lib.lib().ix_moe_pick_low_bm(t * k, 1, e, hd, f) == 160
    w1, w2 = _layer(e, hd, f, 13)
    idx, prob = _routing(t, e, k, hot, 5)
    x = torch.randn(t, hd, generator=_gen(6), device=DEV).to(torch.bfloat16)
    p = permute(idx, prob, e, BM=32)
    experts = [SimpleNamespace(linear_fc1=SimpleNamespace(weight=w1[i]), linear_fc2=SimpleNamespace(weight=w2[i])) for i in range(e)]
    mlp = SimpleNamespace(local_experts=experts, num_local_experts=e)
    for counts in (p.counts, p.counts.long().cpu()):
        out, bias = moe_doors._batched_experts_forward(mlp, x.index_select(0, p.sorted_token.long()), counts, p.permuted_prob)
        assert bias is None and torch.equal(out, experts_forward(x, w1, w2, p))
