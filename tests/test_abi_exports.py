"""The C-ABI library loads without a GPU and exports exactly what include/isoexec_hip.h declares."""

import ctypes
import os
import re

from isoexec_amd import _lib

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HEADER = os.path.join(ROOT, "include", "isoexec_hip.h")


def declared_functions():
    text = open(HEADER).read()
    text = re.sub(r"/\*.*?\*/", "", text, flags=re.S)
    return re.findall(r"^\s*(?:const\s+)?[a-z_0-9]+\*?\s+\*?(ix_[a-z0-9_]+)\s*\(", text, flags=re.M)


def test_header_and_binding_table_agree():
    names = declared_functions()
    assert len(names) >= 20 and len(set(names)) == len(names)
    assert set(names) == set(_lib.SIGNATURES), set(names) ^ set(_lib.SIGNATURES)


def test_library_exports_every_declared_symbol():
    handle = ctypes.CDLL(_lib.LIB_PATH)
    for name in declared_functions():
        assert hasattr(handle, name), name


def test_host_only_entry_points():
    h = _lib.lib()
    assert h.ix_abi_version() == 3 and h.ix_arch_tag() == b"gfx950"
    assert h.ix_moe_max_tiles(16384, 8, 128, 256) == 16384 * 8 // 256 + 128
    assert h.ix_moe_pick_bm(16384, 8, 128) == 256 and h.ix_moe_pick_bm(1, 8, 128) == 32
    assert h.ix_logprob_workspace_bytes(4, 151936, 8) == 4 * (19 + 40 + 2) * 4
    assert h.ix_logprob_workspace_bytes(4, 151937, 8) == 0


def test_a_decode_step_is_described_by_sixteen_numbers():
    """``IxDecodeDims`` as callers of this ABI version lay it out; what lies behind it in memory is not read."""
    dims = (ctypes.c_int64 * 18)(4, 2, 512, 1024, 256, 2, 4, 128, 4, 2, 128, 16, 4, 256, 0, 1)
    need = _lib.lib().ix_decode_step_workspace_bytes(ctypes.addressof(dims))
    assert need > 0
    dims[16] = dims[17] = -1
    assert _lib.lib().ix_decode_step_workspace_bytes(ctypes.addressof(dims)) == need


def test_gemm_tile_choice_is_a_host_decision_with_sane_answers():
    """ix_gemm_bf16_n_tiles reports the row-max parts of the tile shape that would run: forced shapes give
    ceil(N / width), twice that for the four-wave 256 x 256 tile in any of its forms (one part per wave column); the
    automatic choice takes the big square tile for a large product, a 128-wide tile for the router's 128-column
    product, and a narrow tile when there are few rows and few columns."""
    h = _lib.lib()
    widths = {1: (256, 1), 2: (128, 1), 3: (256, 1), 4: (256, 2), 5: (256, 1), 6: (32, 1), 7: (256, 2), 8: (256, 2)}
    for tile, (bn, per_tile) in widths.items():
        for n in (1, 32, 128, 129, 2048, 151936):
            assert h.ix_gemm_bf16_n_tiles(4096, n, 4096, tile) == per_tile * -(-n // bn), (tile, n)
    assert h.ix_gemm_bf16_n_tiles(4096, 151936, 4096, 0) == 2 * -(-151936 // 256)  # LM head: the four-wave 256-wide tile
    assert h.ix_gemm_bf16_n_tiles(163840, 128, 2048, 0) == 1                       # gating product: one 128-wide column
    assert h.ix_gemm_bf16_n_tiles(64, 2048, 2048, 0) == 2048 // 32                 # decode projection: 64 x 32 tiles
    assert h.ix_gemm_bf16_n_tiles(64, 12352, 2048, 0) == 12352 // 32               # wide decode projection: the same
    assert h.ix_gemm_bf16_n_tiles(256, 12352, 2048, 0) in (-(-12352 // 128), -(-12352 // 256), 2 * -(-12352 // 256))  # 256 rows: wider tiles
    assert h.ix_gemm_bf16_n_tiles(0, 0, 4096, 0) == 0


def test_product_path_has_no_cpu_fallback():
    import pytest
    import torch

    from isoexec_amd.ops.mm.mm_hip import linear_nt
    from isoexec_amd.ops.norms.fused_outnorm import fused_rms_norm_gamma

    x = torch.zeros(2, 64, dtype=torch.bfloat16)
    with pytest.raises(_lib.IsoExecLibraryError):
        fused_rms_norm_gamma(x, torch.zeros(64, dtype=torch.bfloat16), 1e-6)
    with pytest.raises(_lib.IsoExecLibraryError):
        linear_nt(x, x)


def test_product_never_imports_the_oracle():
    pkg = os.path.join(ROOT, "skyrl-isoexec_amd")
    for base, _dirs, files in os.walk(pkg):
        for f in files:
            if f.endswith((".py", ".hip", ".h")):
                text = open(os.path.join(base, f)).read()
                assert "from oracle" not in text and "import oracle" not in text, os.path.join(base, f)
