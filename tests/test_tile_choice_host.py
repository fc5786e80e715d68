"""Which tile a product's sizes choose, on the host: the lines between the bands and the other shapes, and the
height of an expert tile."""
import pytest

from isoexec_amd import _lib


@pytest.mark.parametrize("m,n,k,tile_width,parts", [
    (65, 28672, 4096, 128, 1), (100, 28672, 4096, 128, 1), (128, 32000, 4096, 128, 1),  # fewer bands than CUs: 128 x 128
    (100, 40960, 2048, 256, 4), (192, 65536, 1024, 256, 4), (300, 40000, 768, 256, 4), (513, 151936, 4096, 256, 4),  # bands
    (64, 151936, 4096, 128, 1), (256, 151936, 4096, 256, 2),  # up to 64 rows; a whole 256-row tile
    (16, 151936, 2048, 32, 1), (17, 151936, 2048, 128, 1), (8, 200000, 2048, 32, 1), (9, 200000, 2048, 128, 1),  # rows 4 KiB apart
    (7, 80000, 2048, 32, 1), (7, 65536, 2048, 128, 1), (7, 250000, 2048, 128, 1), (7, 151936, 1984, 128, 1)])
def test_dense_tiles(m, n, k, tile_width, parts):
    assert _lib.lib().ix_gemm_bf16_n_tiles(m, n, k, 0) == parts * ((n + tile_width - 1) // tile_width)


@pytest.mark.parametrize("mean,plain,packed", [(15, 32, 32), (23, 128, 64), (24, 96, 96), (70, 96, 96), (71, 160, 160), (126, 160, 160),
                                               (127, 192, 192), (154, 192, 192), (155, 256, 256), (239, 256, 256),
                                               (240, 256, 256), (400, 256, 256)])
def test_expert_tiles(mean, plain, packed):
    pick = _lib.lib().ix_moe_pick_bm_shape
    assert pick(16 * mean, 8, 128, 2048, 768, 0) == plain and pick(16 * mean, 8, 128, 2048, 768, 1) == packed


@pytest.mark.parametrize("T,k,E,hd,f,low", [
    (16 * 239, 8, 128, 2048, 768, 0), (16 * 240, 8, 128, 2048, 768, 160), (16 * 289, 8, 128, 2048, 768, 160),
    (16 * 290, 8, 128, 2048, 768, 192), (16 * 399, 8, 128, 2048, 768, 192), (16 * 400, 8, 128, 2048, 768, 0),
    (2400, 4, 32, 4096, 2048, 0), (256, 1, 1, 2048, 131072, 0), (257, 1, 1, 1024, 131072, 160), (4000, 8, 128, 2048, 700, 0)])
def test_the_lower_of_two_heights(T, k, E, hd, f, low):
    assert _lib.lib().ix_moe_pick_low_bm(T, k, E, hd, f) == low


@pytest.mark.parametrize("T,k,E,hd,f,packed,rows", [
    (1024, 2, 64, 2048, 2048, 0, 96), (1024, 2, 64, 2048, 2048, 1, 64), (1280, 2, 64, 2048, 2048, 1, 96),  # long packed streams
    (1024, 2, 64, 2048, 1024, 0, 128), (640, 4, 32, 2048, 2048, 0, 128), (2400, 4, 32, 4096, 2048, 0, 256),  # two turns of workgroups
    (256, 1, 1, 2048, 131072, 0, 256),  # one token tile
    (1024, 2, 64, 896, 2048, 0, 128), (1024, 2, 64, 2048, 2000, 0, 128)])  # sizes that bands do not serve
def test_expert_tiles_of_other_layers(T, k, E, hd, f, packed, rows):
    assert _lib.lib().ix_moe_pick_bm_shape(T, k, E, hd, f, packed) == rows
