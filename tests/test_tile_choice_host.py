"""Which tile a product's sizes choose, on the host: the lines between the bands and the other shapes."""
import pytest

from isoexec_amd import _lib


@pytest.mark.parametrize("m,n,k,tile_width,parts", [
    (65, 28672, 4096, 128, 1), (100, 28672, 4096, 128, 1), (128, 32000, 4096, 128, 1),  # fewer bands than CUs: 128 x 128
    (100, 40960, 2048, 256, 4), (192, 65536, 1024, 256, 4), (300, 40000, 768, 256, 4), (513, 151936, 4096, 256, 4),  # bands
    (64, 151936, 4096, 128, 1), (256, 151936, 4096, 256, 2)])  # up to 64 rows; a whole 256-row tile
def test_dense_tiles(m, n, k, tile_width, parts):
    assert _lib.lib().ix_gemm_bf16_n_tiles(m, n, k, 0) == parts * ((n + tile_width - 1) // tile_width)
