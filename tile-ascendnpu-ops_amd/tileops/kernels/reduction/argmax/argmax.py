"""ArgreduceKernel: row-wise argmax / argmin returning int64 on gfx950.

Reference class: examples/TileOPs/tileops/kernels/reduction/argmax/argmax.py:89-219.
Semantics are torch.argmax / torch.argmin: first occurrence among equal
values, NaN counts as the extreme value.  The launch is wrapped in the
``tileops::argreduce_fwd`` custom op (reference: ``npub::argreduce_fwd``).
Device code in csrc/reduction.hip: row_reduce_kernel, short_row_kernel and
merge_partials_kernel<T, 1|2, ...>, col_reduce_kernel over other dims.
"""

from typing import Optional

import torch

from tileops import _native
from tileops.kernels.kernel_base import Kernel

__all__ = ["ArgreduceKernel"]

_ARGREDUCE_KINDS = {"argmax", "argmin"}


def _argreduce_fwd_launch(M: int, N: int, op_kind: str, x: torch.Tensor) -> torch.Tensor:
    y = torch.empty((M,), dtype=torch.int64, device=x.device)
    op = _native.ARGMIN if op_kind == "argmin" else _native.ARGMAX
    _native.check(_native.reduce_rows(op, x, y, M, N), "tileops_reduce_fwd")
    return y


_argreduce_fwd = torch.library.custom_op("tileops::argreduce_fwd", mutates_args=())(_argreduce_fwd_launch)


@_argreduce_fwd.register_fake
def _(M: int, N: int, op_kind: str, x: torch.Tensor) -> torch.Tensor:
    return torch.empty((M,), dtype=torch.int64, device=x.device)


def _argreduce_axis_launch(
    outer: int, n: int, inner: int, ends: bool, op_kind: str, x: torch.Tensor
) -> torch.Tensor:
    y = torch.empty((n if ends else outer * inner,), dtype=torch.int64, device=x.device)
    op = _native.ARGMIN if op_kind == "argmin" else _native.ARGMAX
    _native.check(
        _native.reduce_axis(op, x, y, outer, n, inner, ends), "tileops_reduce_axis_fwd")
    return y


_argreduce_axis = torch.library.custom_op("tileops::argreduce_axis_fwd", mutates_args=())(_argreduce_axis_launch)


@_argreduce_axis.register_fake
def _(outer, n, inner, ends, op_kind, x):
    return torch.empty((n if ends else outer * inner,), dtype=torch.int64, device=x.device)


class ArgreduceKernel(Kernel):
    """Argmax / argmin forward kernel; output is always int64.

    Args:
        M: Number of rows.
        N: Reduction length.
        op_kind: ``"argmax"`` or ``"argmin"``.
        dtype: float32, float16 or bfloat16.
        config: Optional config override.
        device_index: Accepted for API compatibility.
    """

    profile_kernel_name = r"tileops(?:::|\d+)(row_reduce|short_row|col_reduce|merge_partials)_kernel"

    def __init__(
        self,
        M: int,
        N: int,
        op_kind: str,
        dtype: torch.dtype,
        config: Optional[dict] = None,
        device_index: Optional[int] = None,
    ):
        super().__init__()
        if op_kind not in _ARGREDUCE_KINDS:
            raise ValueError(
                f"Unsupported op_kind '{op_kind}'. Expected one of {sorted(_ARGREDUCE_KINDS)}."
            )
        self.M = M
        self.N = N
        self.op_kind = op_kind
        self.dtype = dtype
        self.device_index = device_index
        self.init_config(config)

    @property
    def default_config(self) -> dict:
        if self.N == 0:
            raise ValueError(
                "Reduction dimension is empty (N=0). "
                "argmax/argmin over an empty dimension is undefined."
            )
        # as LogSumExpKernel: what rows of middling number and length run with
        return {"wavefronts_per_row": 1 if self.M >= 3072 else 4, "packs_in_flight": 4}

    def forward(self, x: torch.Tensor) -> torch.Tensor:
        _native.require_device(x)
        self.check_tensor("x", x, dtype=self.dtype, shape=(self.M, self.N))
        x = x.contiguous()
        if _native.eager(x):
            return _argreduce_fwd_launch(self.M, self.N, self.op_kind, x)
        return _argreduce_fwd(self.M, self.N, self.op_kind, x)

    def reduce_axis(
        self, x: torch.Tensor, outer: int, n: int, inner: int, ends: bool
    ) -> torch.Tensor:
        """The reduction of contiguous ``x.view(outer, n, inner)`` over n (or, with
        ``ends``, over outer and inner), flat like ``forward``'s result."""
        _native.require_device(x)
        self.check_tensor("x", x, dtype=self.dtype, numel=self.M * self.N)
        if outer * n * inner != self.M * self.N or not x.is_contiguous():
            raise ValueError(f"{type(self).__name__}: expected a contiguous [{outer}, {n}, {inner}]")
        fwd = _argreduce_axis_launch if _native.eager(x) else _argreduce_axis
        return fwd(outer, n, inner, ends, self.op_kind, x)
