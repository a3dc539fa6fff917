"""Multi-dim reduction shape helpers (device independent).

Same contract as the reference's examples/TileOPs/tileops/ops/_multidim.py:22-94:
``normalize_dim`` canonicalises and validates dims, ``flatten_for_multidim``
moves the reduced dims last and flattens to ``[*kept, reduced]``, and
``restore_multidim_shape`` maps the ``(M,)`` result back.
"""

from __future__ import annotations

from math import prod
from typing import Literal, Union

import torch

__all__ = [
    "EmptyDimPolicy",
    "flatten_for_multidim",
    "normalize_dim",
    "restore_multidim_shape",
    "strided_form",
]

EmptyDimPolicy = Literal["reject", "full", "noop"]


def normalize_dim(
    dim: Union[int, list[int], None],
    ndim: int,
    *,
    empty_dim_policy: EmptyDimPolicy = "reject",
) -> list[int]:
    if dim is None:
        return list(range(ndim))
    dims = [dim] if isinstance(dim, int) else list(dim)
    if not dims:
        if empty_dim_policy == "full":
            return list(range(ndim))
        if empty_dim_policy == "noop":
            return []
        raise ValueError(
            "dim=[] is not supported by this op; pass "
            'empty_dim_policy="full" to opt in to full-reduction '
            'or empty_dim_policy="noop" to opt in to the identity contract.'
        )
    out = []
    for d in dims:
        if d < -ndim or d >= ndim:
            raise IndexError(
                f"Dimension out of range (expected to be in range of "
                f"[{-ndim}, {ndim - 1}], but got {d})"
            )
        out.append(d % ndim)
    if len(set(out)) != len(out):
        raise ValueError(f"Duplicate dims in reduction: {dims}")
    return sorted(out)


def strided_form(x: torch.Tensor, dims: list[int]) -> "tuple[int, int, int, bool] | None":
    """``(outer, n, inner, ends)`` when the reduction of ``x`` over ``dims`` (sorted)
    is one over the middle (``ends`` False) or the two outer dims (``ends`` True) of
    ``x.view(outer, n, inner)`` that the kernels read without a copy; None otherwise.

    Below 64 neighbouring columns (or, for ``ends``, rows of 64 elements) the
    strided reads leave most of a wavefront idle and the copy is kept; ``ends``
    merges ``outer`` partials per output on one wavefront, which bounds it.  A
    column workgroup has a slice to itself, so that many small slices, of less
    than 64 packs, are copied too (us, as they lie and copied: LogSumExp bf16
    [131072, 4, 64] 240 and 122, [16384, 4, 64] 36.7 and 24.0, [2048, 4, 64] 6.9 and
    8.3, [16384, 16, 64] 55.5 and 53.5, [16384, 8, 128] 48.8 and 55.0).  As
    on the general path at most 2^31 - 1 elements are reduced to one, and the
    entry point takes each of the three sizes below 2^31.
    """
    if not x.is_contiguous() or x.numel() == 0 or not dims:
        return None
    shape, lo, hi = x.shape, dims[0], dims[-1]
    if hi - lo + 1 == len(dims):  # one run of reduced dims
        outer, n, inner = prod(shape[:lo]), prod(shape[lo:hi + 1]), prod(shape[hi + 1:])
        if inner < 64 or max(outer, n, inner) >= 2**31:
            return None
        if outer >= 16384 and n * inner * x.dtype.itemsize < 64 * 16:
            return None
        return outer, n, inner, False
    kept = [i for i in range(lo, hi + 1) if i not in dims]
    if lo == 0 and hi == x.ndim - 1 and kept[-1] - kept[0] + 1 == len(kept):
        outer, n = prod(shape[:kept[0]]), prod(shape[kept[0]:kept[-1] + 1])
        inner = prod(shape[kept[-1] + 1:])
        if inner < 64 or max(n, outer * inner) >= 2**31 or outer > 16384:
            return None
        return outer, n, inner, True
    return None


def flatten_for_multidim(
    x: torch.Tensor, dims: list[int]
) -> tuple[torch.Tensor, torch.Size, list[int]]:
    orig_shape = x.shape
    kept = [i for i in range(x.ndim) if i not in dims]
    x = x.permute(kept + list(dims)).contiguous()
    kept_shape = [orig_shape[i] for i in kept]
    reduced = 1
    for d in dims:
        reduced *= orig_shape[d]
    return x.reshape(kept_shape + [reduced] if kept_shape else [1, reduced]), orig_shape, kept


def restore_multidim_shape(
    y: torch.Tensor, orig_shape: torch.Size, dims: list[int], keepdim: bool
) -> torch.Tensor:
    if keepdim:
        shape = list(orig_shape)
        for d in dims:
            shape[d] = 1
        return y.reshape(shape)
    shape = [orig_shape[i] for i in range(len(orig_shape)) if i not in dims]
    return y.squeeze() if not shape else y.reshape(shape)
