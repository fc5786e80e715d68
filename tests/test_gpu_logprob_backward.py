"""Gradient kernel of the sampled logprob against the eager expression in float64, at the edges of its segments."""

import pytest
import torch

from _util import cpu_gen

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("vocab", [8, 24, 4099, 8192, 8200, 16384 + 8, 24577])
def test_sampled_backward(vocab, dtype):
    """Whole and ragged segments of 8192 columns, an odd vocabulary (element path), strided rows, targets at both ends and
    outside. Bound: expf and one product, 4 fp32 units of the float64 value, and half a unit of bf16 where it is stored so."""
    from isoexec_amd.ops.logprobs.rowinv import sampled_backward

    g = cpu_gen(vocab)
    rows, pitch = 5, vocab + (8 if vocab % 8 == 0 else 3)
    x = (3 * torch.randn(rows, pitch, generator=g)).to(dtype).to(DEV)[:, :vocab]
    t = torch.tensor([0, vocab - 1, vocab // 2, -1, vocab], device=DEV)
    u = torch.randn(rows, generator=g).to(DEV)
    lse = torch.logsumexp(x.double(), 1).float()
    got = sampled_backward(x, t, u, lse)
    valid = (t >= 0) & (t < vocab)
    ud = torch.where(valid, u, 0.0).double()
    want = -ud[:, None] * torch.exp(x.double() - lse.double()[:, None])
    want.scatter_add_(1, torch.where(valid, t, 0)[:, None], ud[:, None])
    assert got.dtype is dtype and got.shape == (rows, vocab)
    scale = want.abs() + (ud.abs()[:, None] if vocab < 64 else 0) + torch.zeros_like(want).scatter_(1, t.clamp(0, vocab - 1)[:, None], ud.abs()[:, None])
    # the argument x - lse is rounded to fp32 as in the eager expression: up to half a unit of its size, times the value
    arg = (x.double() - lse.double()[:, None]).abs()
    tol = scale * (4 + arg) * 2.0 ** -23 + (want.abs() * 2.0 ** -8 if dtype is torch.bfloat16 else 0) + 1e-37
    assert bool(((got.double() - want).abs() <= tol).all())


def test_gradient_through_the_function_equals_the_differentiable_form():
    """The autograd function's gradient is the kernel's; asked for with ``create_graph`` it is the eager expression."""
    from isoexec_amd.ops.logprobs.rowinv import _RowInvSampledLogprob

    g = cpu_gen(2)
    x = torch.randn(2, 7, 4096, generator=g).to(DEV).requires_grad_(True)
    t = torch.randint(0, 4096, (2, 7), generator=g).to(DEV)
    u = torch.randn(2, 7, generator=g).to(DEV)
    (a,) = torch.autograd.grad(_RowInvSampledLogprob.apply(x, t, 8), x, u)
    (b,) = torch.autograd.grad(_RowInvSampledLogprob.apply(x, t, 8), x, u, create_graph=True)
    assert b.requires_grad and float((a - b.detach()).abs().max()) <= 2.0 ** -22 * float(a.abs().max())


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_a_gradient_larger_than_the_caches_equals_its_rows_taken_by_themselves(dtype):
    """From 256 MiB of logits both streams go past the caches: the bits of calls below that line."""
    from isoexec_amd.ops.logprobs.rowinv import sampled_backward

    vocab = 16384 + 8
    rows = (256 << 20) // (vocab * dtype.itemsize) + 2
    x = torch.randn(rows, vocab, generator=torch.Generator(device=DEV).manual_seed(1), device=DEV).to(dtype)
    t = torch.randint(-1, vocab + 1, (rows,), generator=cpu_gen(3)).to(DEV)
    u = torch.randn(rows, generator=cpu_gen(4)).to(DEV)
    lse = torch.logsumexp(x.float(), 1)
    whole = sampled_backward(x, t, u, lse)
    half = rows // 2
    parts = [sampled_backward(x[a:b], t[a:b], u[a:b], lse[a:b]) for a, b in ((0, half), (half, rows))]
    assert torch.equal(whole, torch.cat(parts))


def test_strided_targets_and_an_expanded_upstream(monkeypatch):
    """Targets that are a view of a wider label tensor, and the upstream of a ``.sum()`` (one element, expanded): both are
    copied for the kernel, and the gradient is the one of contiguous operands."""
    from isoexec_amd.ops.logprobs.rowinv import rowinv_sampled_logprobs

    monkeypatch.setenv("SKYRL_ISOEXEC", "1")
    g = cpu_gen(5)
    x = torch.randn(2, 300, 512, generator=g).to(DEV).requires_grad_(True)
    labels = torch.randint(0, 512, (2, 300, 2), generator=g).to(DEV)
    call = lambda t: rowinv_sampled_logprobs(x, t, vocab_start_index=0, vocab_end_index=512, group=None,
                                             src_dtype=torch.float32, reference=None)
    (want,) = torch.autograd.grad(call(labels[:, :, 0].contiguous()), x, torch.ones(2, 300, device=DEV))
    (got,) = torch.autograd.grad(call(labels[:, :, 0]).sum(), x)
    assert torch.equal(got, want)
