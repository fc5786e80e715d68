"""Operands that a wrapper copies to a contiguous layout stay alive until the library has been called: two temporaries in one
call may otherwise share one allocation, and the kernel reads the second in the place of the first. The library is replaced
by a stub that reads the memory behind the pointers it is handed, on the CPU."""

import ctypes

import pytest
import torch

ROWS = 64  # small blocks: the allocator hands a freed one straight out again


class Stub:
    """Every entry point returns ``values.get(name, 0)``; the first call of ``name`` copies ``sizes`` bytes behind the pointer
    arguments at the given positions."""

    def __init__(self, name, sizes, **values):
        self.name, self.sizes, self.values, self.seen = name, sizes, values, None

    def __getattr__(self, entry):
        def call(*args):
            if entry == self.name:
                self.seen = {i: ctypes.string_at(args[i], n) for i, n in self.sizes.items()}
            return self.values.get(entry, 0)

        return call


def as_bytes(t):
    t = t.contiguous()
    return ctypes.string_at(t.data_ptr(), t.numel() * t.element_size())


@pytest.fixture
def stub(monkeypatch):
    from isoexec_amd import _lib

    def install(s):
        monkeypatch.setattr(_lib, "lib", lambda: s)
        monkeypatch.setattr(_lib, "require_device", lambda *t: None)
        monkeypatch.setattr(_lib, "current_stream", lambda device=None: 0)
        return s

    return install


def strided(t):
    """The same values, every other element of a wider tensor."""
    return torch.stack([t, t], dim=-1)[..., 0]


def test_logprob_gradient(stub):
    from isoexec_amd.ops.logprobs.rowinv import sampled_backward

    x = torch.randn(ROWS, 8)
    t, u, lse = torch.arange(ROWS) % 8, torch.ones(1).expand(ROWS), torch.randn(ROWS)
    s = stub(Stub("ix_logprob_rowinv_backward", {5: 8 * ROWS, 6: 4 * ROWS, 7: 4 * ROWS}))
    assert sampled_backward(x, strided(t), u, strided(lse)) is not None
    assert s.seen == {5: as_bytes(t), 6: as_bytes(u), 7: as_bytes(lse)}


def test_permutation(stub):
    from isoexec_amd.ops.moe.moe_hip import permute

    idx, prob = torch.randint(0, 4, (ROWS, 2), dtype=torch.int32), torch.rand(ROWS, 2)
    sizes = {0: 8 * ROWS, 1: 8 * ROWS}
    for entry, kw in (("ix_moe_permute", {}), ("ix_moe_permute_static", {"static_scratch": True})):
        s = stub(Stub(entry, sizes, ix_moe_max_tiles=8, ix_moe_permute_scratch_ints=8))
        permute(strided(idx), strided(prob), 4, BM=32, **kw)
        assert s.seen == {0: as_bytes(idx), 1: as_bytes(prob)}, entry


def test_experts(stub):
    from isoexec_amd.ops.moe.moe_hip import experts_forward, permute

    w1, w2 = torch.randn(4, 16, 16).bfloat16(), torch.randn(4, 16, 16).bfloat16()[:, :, :8].contiguous()
    s = stub(Stub("ix_moe_experts_tile", {4: w1.numel() * 2, 5: w2.numel() * 2}, ix_moe_max_tiles=8,
                  ix_moe_permute_scratch_ints=8))
    p = permute(torch.zeros(ROWS, 1, dtype=torch.int32), torch.ones(ROWS, 1), 4, BM=32)
    experts_forward(torch.randn(ROWS, 16).bfloat16(), strided(w1), strided(w2), p)
    assert s.seen == {4: as_bytes(w1), 5: as_bytes(w2)}


def test_attention(stub):
    from isoexec_amd.ops.attention.varlen_attn import varlen_attention

    q = torch.randn(ROWS, 2, 128).bfloat16()
    kv = torch.randn(2 * ROWS, 1, 128).bfloat16()
    start, pos = torch.arange(ROWS), torch.arange(ROWS, dtype=torch.int32)
    s = stub(Stub("ix_attn_varlen", {7: 8 * ROWS, 8: 4 * ROWS}))
    varlen_attention(q, kv, kv, torch.arange(ROWS + 1, dtype=torch.int32), 1, kv_start=strided(start), q_pos0=strided(pos))
    assert s.seen == {7: as_bytes(start), 8: as_bytes(pos)}


def test_decode_preparation(stub):
    from isoexec_amd.ops.gdn.gdn_ops import decode_prep

    n, hv, d = 2, ROWS, 2 * 128 + ROWS * 128
    bf = lambda *shape: torch.randn(*shape).bfloat16()
    a_log, dt = torch.randn(hv), torch.randn(hv)
    s = stub(Stub("ix_gdn_decode_prep", {8: 4 * hv, 9: 4 * hv}))
    decode_prep(bf(n, d), bf(n, hv), bf(n, hv), bf(d, 4), None, strided(a_log), strided(dt), bf(3, d, 3),
                torch.ones(n, dtype=torch.int32), H=1, K=128, HV=hv, V=128)
    assert s.seen == {8: as_bytes(a_log), 9: as_bytes(dt)}
