"""Batch-invariant dense matmul on the fixed-K-order MFMA kernel.

Counterpart of the reference's global ``aten::mm/addmm/bmm`` override
(``ops/moe/moe_batch_invariant.py:422-473``) and of ``ops/mm/mm_cublaslt.py``: every
``F.linear`` of the model reaches one kernel whose per-element accumulation order does not
depend on M. On ROCm the dispatch key is still "CUDA".
"""

from __future__ import annotations

import torch

from ... import _lib

_LIBRARY = None
_COUNTS = {"mm": 0, "addmm": 0, "bmm": 0, "declined": 0, "operand_copies": 0}


def stats() -> dict:
    """Calls served per primitive since import, calls handed to the stock kernel, operands copied to reach the
    kernel's K-contiguous layout."""
    return dict(_COUNTS)


def reset_stats() -> None:
    for key in _COUNTS:
        _COUNTS[key] = 0


DECODE_ROWS = 64  # the streaming form serves products of at most this many rows


class PackedWeight:
    """A weight ``[N, K]`` and its fragment-packed copy for products of at most ``DECODE_ROWS`` rows. The copy is made
    by ``pack_nt_decode`` and is as large as the weight; it has to be made again when the weight changes. ``footprint``: the
    bytes the owner knows to be read between two products with this weight (0: nothing known; a cache choice, not a bit)."""

    __slots__ = ("weight", "packed", "footprint")

    def __init__(self, weight: torch.Tensor, packed: torch.Tensor, footprint: int = 0):
        self.weight, self.packed, self.footprint = weight, packed, footprint

    @property
    def shape(self):
        return self.weight.shape


def pack_nt_decode(weight: torch.Tensor):
    """``PackedWeight`` for ``weight [N, K]`` (bf16, rows K-contiguous), or ``None`` for a shape the streaming form does
    not serve (N a multiple of 32, K in {1024, 2048, 3072, 4096})."""
    _lib.require_device(weight)
    if weight.dtype is not torch.bfloat16 or weight.ndim != 2 or weight.stride(1) != 1:
        return None
    n, k = weight.shape
    L = _lib.lib()
    if not L.ix_gemm_decode_serves_shape(n, k):
        return None
    packed = torch.empty(n * k, dtype=torch.bfloat16, device=weight.device)
    rc = _lib.check(L.ix_gemm_pack_decode(weight.data_ptr(), weight.stride(0), packed.data_ptr(), n, k,
                                          _lib.current_stream(weight.device)), "ix_gemm_pack_decode")
    return PackedWeight(weight, packed) if rc == _lib.IX_OK else None


def linear_nt_decode(x: torch.Tensor, packed: PackedWeight):
    """``x [M <= 64, K] @ weight^T`` from the packed copy (bf16 out, same bits as ``linear_nt``); ``None`` if declined."""
    _lib.require_device(x, packed.packed)
    if x.dtype is not torch.bfloat16 or x.ndim != 2 or x.stride(1) != 1 or x.shape[1] != packed.weight.shape[1]:
        return None
    m, k = x.shape
    if m > DECODE_ROWS:
        return None
    n = packed.weight.shape[0]
    out = torch.empty(m, n, dtype=torch.bfloat16, device=x.device)
    rc = _lib.check(
        _lib.lib().ix_gemm_bf16_nt_decode_footprint(x.data_ptr(), x.stride(0), packed.packed.data_ptr(), out.data_ptr(),
                                                    out.stride(0), m, n, k, packed.footprint,
                                                    _lib.current_stream(x.device)), "ix_gemm_bf16_nt_decode")
    return out if rc == _lib.IX_OK else None


def linear_nt(x: torch.Tensor, weight, bias: torch.Tensor | None = None, *, tile: int = 0,
              out_dtype: torch.dtype = torch.bfloat16, want_row_max: bool = False):
    """``x [M, K] @ weight [N, K]^T (+ bias)``, bf16 operands, fp32 accumulate; ``None`` if declined.

    ``out_dtype=torch.float32`` returns the fp32 accumulator unrounded. ``want_row_max`` also returns
    each row's exact maximum over the N outputs (taken in the kernel's epilogue), as ``(out, row_max)``.
    ``weight`` may be a ``PackedWeight``: a plain product (no bias, bf16 out, no row maximum, tile 0) of at most
    ``DECODE_ROWS`` rows then streams the packed copy; every other call uses the weight itself. Same bits either way.
    """
    if isinstance(weight, PackedWeight):
        if (bias is None and tile == 0 and out_dtype is torch.bfloat16 and not want_row_max
                and 0 < x.shape[0] <= DECODE_ROWS):
            out = linear_nt_decode(x, weight)
            if out is not None:
                return out
        weight = weight.weight
    _lib.require_device(x, weight, bias)
    if x.dtype is not torch.bfloat16 or weight.dtype is not torch.bfloat16:
        return None
    if x.ndim != 2 or weight.ndim != 2 or x.shape[1] != weight.shape[1]:
        raise RuntimeError(f"linear_nt shape mismatch {tuple(x.shape)} x {tuple(weight.shape)}")
    if x.stride(1) != 1 or weight.stride(1) != 1:
        return None
    m, k = x.shape
    n = weight.shape[0]
    out = torch.empty(m, n, dtype=out_dtype, device=x.device)
    if bias is not None and (bias.dtype is not torch.bfloat16 or not bias.is_contiguous()):
        return None
    L = _lib.lib()
    parts = None
    n_parts = 0
    if want_row_max:
        n_parts = int(L.ix_gemm_bf16_n_tiles(m, n, k, tile))
        parts = torch.empty(m, n_parts, dtype=torch.float32, device=x.device)
    stream = _lib.current_stream(x.device)
    rc = _lib.check(
        L.ix_gemm_bf16_nt(x.data_ptr(), x.stride(0), weight.data_ptr(), weight.stride(0), _lib.ptr(bias),
                          out.data_ptr(), _lib.dtype_code(out_dtype), out.stride(0), m, n, k, tile,
                          _lib.ptr(parts), n_parts, stream), "ix_gemm_bf16_nt")
    if rc != _lib.IX_OK:
        return None
    if not want_row_max:
        return out
    row_max = torch.empty(m, dtype=torch.float32, device=x.device)
    if m:
        _lib.check(L.ix_rowmax_reduce(parts.data_ptr(), n_parts, n_parts, m, row_max.data_ptr(), stream),
                   "ix_rowmax_reduce")
    return out, row_max


def router_gemm(x: torch.Tensor, weight: torch.Tensor):
    """Router gating logits in fp32. A bf16 router weight (exactly what an fp32 cast of a bf16
    checkpoint holds) multiplies exactly in the bf16 MFMA and is accumulated in fp32, so the bf16
    core with an fp32 store IS the fp32 gating product; an fp32 weight takes the fp32 kernel."""
    if weight.dtype is torch.bfloat16 and x.dtype is torch.bfloat16:
        return linear_nt(x, weight, out_dtype=torch.float32)
    return linear_f32_nt(x, weight.float())


def linear_f32_nt(x: torch.Tensor, weight: torch.Tensor):
    """Router gating: ``x [M, K]`` (bf16 or fp32) ``@ weight [N, K]^T`` (fp32) -> fp32."""
    _lib.require_device(x, weight)
    if weight.dtype is not torch.float32 or x.stride(1) != 1 or weight.stride(1) != 1:
        return None
    m, k = x.shape
    n = weight.shape[0]
    out = torch.empty(m, n, dtype=torch.float32, device=x.device)
    rc = _lib.check(
        _lib.lib().ix_gemm_f32_nt(x.data_ptr(), _lib.dtype_code(x.dtype), x.stride(0), weight.data_ptr(),
                                  weight.stride(0), out.data_ptr(), out.stride(0), m, n, k,
                                  _lib.current_stream(x.device)), "ix_gemm_f32_nt")
    return out if rc == _lib.IX_OK else None


def _as_nt(b: torch.Tensor):
    """``b [K, N]`` as a K-contiguous ``[N, K]`` matrix: free for the transposed view of a ``[N, K]`` weight (what
    ``F.linear`` hands to ``aten::mm``); a ``[K, N]`` operand that is itself row-major (a backward-pass product) is
    copied, and the copy is counted in ``stats()["operand_copies"]``."""
    bt = b.transpose(-1, -2)
    if bt.stride(-1) == 1:
        return bt
    _COUNTS["operand_copies"] += 1
    return bt.contiguous()


def _rows(a: torch.Tensor):
    if a.stride(-1) == 1:
        return a
    _COUNTS["operand_copies"] += 1
    return a.contiguous()


def mm_batch_invariant(a: torch.Tensor, b: torch.Tensor):
    """``a [M, K] @ b [K, N]`` on the fixed-order kernels, or ``None`` for a signature they do not serve."""
    if a.ndim != 2 or b.ndim != 2 or not a.is_cuda or not b.is_cuda:
        return None
    if a.dtype is torch.bfloat16 and b.dtype is torch.bfloat16:
        return linear_nt(_rows(a), _as_nt(b))
    if a.dtype is torch.float32 and b.dtype is torch.float32:
        return linear_f32_nt(_rows(a), _as_nt(b))
    return None


def addmm_batch_invariant(bias, a, b, *, beta=1, alpha=1):
    """``bias [N] + a @ b`` (bf16, alpha = beta = 1: what ``F.linear`` with a bias dispatches), else ``None``."""
    if beta != 1 or alpha != 1 or bias.ndim != 1 or a.ndim != 2 or b.ndim != 2:
        return None
    if not (a.dtype is b.dtype is bias.dtype is torch.bfloat16) or bias.shape[0] != b.shape[1]:
        return None
    return linear_nt(_rows(a), _as_nt(b), bias.contiguous())


def bmm_batch_invariant(a: torch.Tensor, b: torch.Tensor):
    """``a [B, M, K] @ b [B, K, N]``: ONE launch over the batch, every product computed exactly as ``mm`` computes
    it (same bits as a loop of ``mm_batch_invariant``); ``None`` for a signature the kernel does not serve."""
    if a.ndim != 3 or b.ndim != 3 or a.dtype is not torch.bfloat16 or b.dtype is not torch.bfloat16:
        return None
    if not a.is_cuda or a.shape[0] != b.shape[0] or a.shape[2] != b.shape[1]:
        return None
    ar, bt = _rows(a), _as_nt(b)          # [B, M, K], [B, N, K], rows K-contiguous
    if ar.stride(1) < ar.shape[2] or bt.stride(1) < bt.shape[2]:
        return None
    B, M, K = ar.shape
    N = bt.shape[1]
    out = torch.empty(B, M, N, dtype=torch.bfloat16, device=a.device)
    if B == 0 or M == 0:
        return out
    rc = _lib.check(
        _lib.lib().ix_gemm_bf16_nt_batched(ar.data_ptr(), ar.stride(1), ar.stride(0), bt.data_ptr(), bt.stride(1),
                                           bt.stride(0), out.data_ptr(), N, M * N, B, M, N, K, 0,
                                           _lib.current_stream(a.device)), "ix_gemm_bf16_nt_batched")
    return out if rc == _lib.IX_OK else None


# ---- the operator override (moe_batch_invariant.py:422-473) -------------------------------------------------------
# aten::mm / addmm / bmm on the device dispatch key are replaced, so every F.linear / torch.matmul of the process
# lands on the fixed-order kernels (matmul and linear are composite: only these three primitives need replacing).
# A signature the kernels do not serve (other dtypes, K or a row pitch that is not a multiple of 8, alpha/beta forms)
# raises by default (``strict=True``): a product that silently took the stock kernel is not batch-invariant, and the
# reference's own notes record that partial coverage of the override broke bitwise parity live. With the explicit
# opt-in ``strict=False`` (a process that also runs products outside the contract, e.g. a backward pass) such a
# signature is handed to the kernel that was registered before, counted under "declined" and named once on stderr;
# ``assert_none_declined()`` then turns the count into a refusal at a point of the caller's choosing.
_STOCK = {}
_STRICT = False
_NAMED = set()


def _fall_through(name, keyset, args, kwargs):
    _COUNTS["declined"] += 1
    sig = (name,) + tuple((tuple(t.shape), str(t.dtype)) for t in args if isinstance(t, torch.Tensor))
    if _STRICT:
        raise RuntimeError(f"[isoexec-amd] {name} override: no batch-invariant kernel for {sig[1:]}")
    if sig not in _NAMED and len(_NAMED) < 32:
        _NAMED.add(sig)
        import sys

        print(f"[isoexec-amd] {name}: {sig[1:]} is not served by the batch-invariant kernels; stock kernel used",
              file=sys.stderr, flush=True)
    return _STOCK[name].call_boxed(keyset, *args, **kwargs)


def _mm_impl(keyset, a, b):
    out = mm_batch_invariant(a, b)
    if out is None:
        return _fall_through("mm", keyset, (a, b), {})
    _COUNTS["mm"] += 1
    return out


def _addmm_impl(keyset, bias, a, b, *, beta=1, alpha=1):
    out = addmm_batch_invariant(bias, a, b, beta=beta, alpha=alpha)
    if out is None:
        return _fall_through("addmm", keyset, (bias, a, b), {"beta": beta, "alpha": alpha})
    _COUNTS["addmm"] += 1
    return out


def _bmm_impl(keyset, a, b):
    out = bmm_batch_invariant(a, b)
    if out is None:
        return _fall_through("bmm", keyset, (a, b), {})
    _COUNTS["bmm"] += 1
    return out


def assert_none_declined(since: int = 0) -> None:
    """Raise if any product was handed to the stock kernel since the count stood at ``since`` (``stats()["declined"]``
    read before the forward): the check a fall-through install owes after every forward under the contract."""
    n = _COUNTS["declined"] - since
    if n > 0:
        raise RuntimeError(f"[isoexec-amd] {n} matrix product(s) ran on the stock kernel, which is not batch-invariant: "
                           f"{sorted(_NAMED)[:8]}")


def install_mm_override(strict: bool = True) -> bool:
    """Route ``aten::mm/addmm/bmm`` on device tensors to the kernels (moe_batch_invariant.py:453-464). ``strict``
    (the default): a signature the kernels do not serve raises; ``strict=False``: it falls through to the stock kernel
    and is counted."""
    global _LIBRARY, _STRICT
    _STRICT = bool(strict)
    if _LIBRARY is not None:
        return True
    _lib.lib()
    for name in ("mm", "addmm", "bmm"):
        _STOCK[name] = torch.library.get_kernel(f"aten::{name}", "CUDA")
    library = torch.library.Library("aten", "IMPL")
    library.impl("mm", _mm_impl, "CUDA", with_keyset=True)
    library.impl("addmm", _addmm_impl, "CUDA", with_keyset=True)
    library.impl("bmm", _bmm_impl, "CUDA", with_keyset=True)
    _LIBRARY = library
    return True


def uninstall_mm_override() -> None:
    """Remove the override: the kernels registered before serve again."""
    global _LIBRARY
    if _LIBRARY is not None:
        _LIBRARY._destroy()
        _LIBRARY = None
    _STOCK.clear()


def mm_override_installed() -> bool:
    return _LIBRARY is not None
