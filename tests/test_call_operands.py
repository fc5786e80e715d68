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
