"""LogSumExpKernel: row-wise log-sum-exp over an (M, N) tensor on gfx950.

Reference class: examples/TileOPs/tileops/kernels/reduction/logsumexp/logsumexp.py:150-336.
y[i] = max_i + log(sum_j exp(x[i, j] - max_i)) in fp32, rounded to the input
dtype.  Lanes fold a row with online (max, scaled-sum) pairs, in a few lanes of
a wavefront or in several workgroups by the shape, so any N works without host
padding.  The launch is wrapped in the
``tileops::logsumexp_fwd`` custom op (with a fake impl) so ``torch.compile``
can trace through it, as the reference's ``npub::logsumexp_fwd`` did.
Device code in csrc/reduction.hip: row_reduce_kernel, short_row_kernel and
merge_partials_kernel<T, 0, ...>, col_reduce_kernel over other dims.
"""

from typing import Optional

import torch

from tileops import _native
from tileops.kernels.kernel_base import Kernel

__all__ = ["LogSumExpKernel"]


def _logsumexp_fwd_launch(M: int, N: int, x: torch.Tensor) -> torch.Tensor:
    y = torch.empty((M,), dtype=x.dtype, device=x.device)
    _native.check(_native.reduce_rows(_native.LOGSUMEXP, x, y, M, N), "tileops_reduce_fwd")
    return y


_logsumexp_fwd = torch.library.custom_op("tileops::logsumexp_fwd", mutates_args=())(_logsumexp_fwd_launch)


@_logsumexp_fwd.register_fake
def _(M: int, N: int, x: torch.Tensor) -> torch.Tensor:
    return torch.empty((M,), dtype=x.dtype, device=x.device)


def _logsumexp_axis_launch(
    outer: int, n: int, inner: int, ends: bool, x: torch.Tensor
) -> torch.Tensor:
    y = torch.empty((n if ends else outer * inner,), dtype=x.dtype, device=x.device)
    _native.check(
        _native.reduce_axis(_native.LOGSUMEXP, x, y, outer, n, inner, ends), "tileops_reduce_axis_fwd")
    return y


_logsumexp_axis = torch.library.custom_op("tileops::logsumexp_axis_fwd", mutates_args=())(_logsumexp_axis_launch)


@_logsumexp_axis.register_fake
def _(outer, n, inner, ends, x):
    return torch.empty((n if ends else outer * inner,), dtype=x.dtype, device=x.device)


class LogSumExpKernel(Kernel):
    """LogSumExp forward kernel.

    Args:
        M: Number of rows.
        N: Reduction length.
        op_kind: Must be ``"logsumexp"``.
        dtype: float32, float16 or bfloat16.
        config: Optional config override.
        device_index: Accepted for API compatibility (the kernel needs no
            per-device sizing).
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
        if op_kind != "logsumexp":
            raise ValueError(f"Unsupported op_kind '{op_kind}'. Expected 'logsumexp'.")
        self.M = M
        self.N = N
        self.op_kind = op_kind
        self.dtype = dtype
        self.device_index = device_index
        self.init_config(config)

    @property
    def default_config(self) -> dict:
        # what rows of middling number and length run with; the library goes by
        # the shape (plan_rows in csrc/reduction.hip): few long rows take sixteen
        # wavefronts or several workgroups each, short rows part of a wavefront
        return {"wavefronts_per_row": 1 if self.M >= 3072 else 4, "packs_in_flight": 4}

    def forward(self, x: torch.Tensor) -> torch.Tensor:
        _native.require_device(x)
        self.check_tensor("x", x, dtype=self.dtype, shape=(self.M, self.N))
        x = x.contiguous()
        if _native.eager(x):
            return _logsumexp_fwd_launch(self.M, self.N, x)
        return _logsumexp_fwd(self.M, self.N, x)

    def reduce_axis(
        self, x: torch.Tensor, outer: int, n: int, inner: int, ends: bool
    ) -> torch.Tensor:
        """The reduction of contiguous ``x.view(outer, n, inner)`` over n (or, with
        ``ends``, over outer and inner), flat like ``forward``'s result."""
        _native.require_device(x)
        self.check_tensor("x", x, dtype=self.dtype, numel=self.M * self.N)
        if outer * n * inner != self.M * self.N or not x.is_contiguous():
            raise ValueError(f"{type(self).__name__}: expected a contiguous [{outer}, {n}, {inner}]")
        fwd = _logsumexp_axis_launch if _native.eager(x) else _logsumexp_axis
        return fwd(outer, n, inner, ends, x)
