"""Expert GEMMs that stream fragment-packed weights: 64-row tiles and the sizes where a tile's second block of tokens starts
or stops being live, and which tile shape a caller with packed matrices gets."""

import pytest
import torch

from _util import cpu_gen, same_bits

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def make(T, H, E, F, seed):
    g = cpu_gen(seed)
    bf = lambda *s: torch.randn(*s, generator=g).to(torch.bfloat16).to(DEV)
    return bf(T, H), bf(E, 2 * F, H) * 0.02, bf(E, H, F) * 0.02


@pytest.mark.parametrize("counts", [[32, 33, 1, 0], [64, 65, 31, 63], [128, 0, 96, 97]])
@pytest.mark.parametrize("H,F", [(512, 768), (2048, 1024), (4096, 512)])
def test_64_row_tiles_equal_the_ring_tiles(H, F, counts):
    """Rows per expert around 32 and 64 (one live block, two, a second tile), against the 256-row ring tile; H and F cover
    both ring depths."""
    from isoexec_amd.ops.moe.moe_hip import experts_forward, pack_decode, permute

    E, T = len(counts), sum(counts)
    x, w1, w2 = make(T, H, E, F, seed=T + H)
    idx = torch.repeat_interleave(torch.arange(E, dtype=torch.int32), torch.tensor(counts))[torch.randperm(T, generator=cpu_gen(1))]
    idx = idx.view(T, 1).contiguous().to(DEV)
    prob = torch.rand(T, 1, generator=cpu_gen(2)).to(DEV)
    packed = pack_decode(w1, w2)
    want, wi = experts_forward(x, w1, w2, permute(idx, prob, E, BM=256), return_inter=True)
    for bm in (32, 64):
        got, gi = experts_forward(x, w1, w2, permute(idx, prob, E, BM=bm), return_inter=True, packed=packed)
        assert same_bits(gi, wi) and same_bits(got, want), bm


@pytest.mark.parametrize("T", [1, 3, 255, 256, 257, 639, 640, 1407, 1408])
def test_layer_with_packed_matrices_equals_the_layer_without(T):
    """Both sides of every line of the tile choice: 16, 40 and 88 rows per expert are 256, 640 and 1408 tokens of 16 experts,
    one each."""
    from isoexec_amd.ops.moe.moe_hip import moe_ffn_forward, pack_decode

    E, H, F = 16, 512, 512
    x, w1, w2 = make(T, H, E, F, seed=T)
    wr = torch.randn(E, H, generator=cpu_gen(7)).to(torch.bfloat16).to(DEV) * 0.02
    want = moe_ffn_forward(x, wr, w1, w2, 1, pre_softmax=True)
    assert same_bits(moe_ffn_forward(x, wr, w1, w2, 1, pre_softmax=True, packed=pack_decode(w1, w2)), want)
