"""LogSumExpFwdOp and ArgmaxFwdOp against the oracle.

Mirrors tests/ops/test_softmax.py (LogSumExp subset) and tests/ops/test_argmax.py
of the reference: shapes, dims, keepdim, dim=None, non-contiguous input, the
multidim rejection, roofline; argmax indices compared exactly (torch.equal).
Adds special-value rows (all -inf, +inf, NaN, ties, signed zeros).
"""

import numpy as np
import pytest
import torch

from oracle import tileops_oracle as orc
from tests._util import NAMES, assert_close_np, from_np, ref_tolerance, to_np
from tileops import _native
from tileops.kernels.reduction.argmax import ArgreduceKernel
from tileops.kernels.reduction.logsumexp import LogSumExpKernel
from tileops.ops.reduction.argmax import ArgmaxFwdOp
from tileops.ops.reduction.softmax import LogSumExpFwdOp
from tileops.testing.test_base import TestBase
from tileops.workloads.reduction import ArgmaxWorkload, LogSumExpWorkload


def _exact_compare(output, output_ref):
    assert output.dtype == torch.int64 and output_ref.dtype == torch.int64
    assert torch.equal(output, output_ref.to(output.device)), (
        f"mismatches: {(output.cpu() != output_ref.cpu()).sum().item()} / {output.numel()}"
    )


def _lse_ref(x, dim, keepdim=False):
    a = to_np(x)
    dims = [dim] if isinstance(dim, int) else list(dim)
    dims = sorted(d % a.ndim for d in dims)
    kept = [i for i in range(a.ndim) if i not in dims]
    flat = np.transpose(a, kept + dims).reshape([a.shape[i] for i in kept] + [-1])
    y = orc.logsumexp(flat, NAMES[x.dtype])
    if keepdim:
        shape = list(a.shape)
        for d in dims:
            shape[d] = 1
        y = y.reshape(shape)
    return y


class LogSumExpTest(LogSumExpWorkload, TestBase):
    def __init__(self, shape, dtype, dim=-1):
        super().__init__(shape, dtype)
        self.dim = dim

    def ref_program(self, x):
        return from_np(np.asarray(_lse_ref(x, self.dim)), x)


@pytest.mark.gpu
@pytest.mark.parametrize(
    "shape, dim, dtype",
    [
        pytest.param((32, 256), -1, torch.float32, marks=[pytest.mark.smoke]),
        pytest.param((32, 256), -1, torch.float16, marks=pytest.mark.smoke),
        pytest.param((32, 256), -1, torch.bfloat16, marks=pytest.mark.smoke),
        pytest.param((32, 300), -1, torch.float32, marks=pytest.mark.full),
        pytest.param((32, 300), -1, torch.float16, marks=pytest.mark.full),
        pytest.param((32, 300), -1, torch.bfloat16, marks=pytest.mark.full),
        pytest.param((33, 256), -1, torch.float32, marks=pytest.mark.full),
        pytest.param((2, 16, 256), -1, torch.float16, marks=pytest.mark.full),
        pytest.param((4, 32768), -1, torch.float16, marks=pytest.mark.full),
        pytest.param((4, 102400), -1, torch.bfloat16, marks=pytest.mark.full),
        pytest.param((256, 32), 0, torch.float32, marks=pytest.mark.full),
        pytest.param((256, 32), 0, torch.float16, marks=pytest.mark.full),
        pytest.param((8192, 4096), -1, torch.float32, marks=pytest.mark.full),
        pytest.param((4000, 131), -1, torch.float32, marks=pytest.mark.full),
    ],
)
def test_logsumexp_op(shape, dim, dtype):
    test = LogSumExpTest(shape, dtype, dim=dim)
    atol, rtol = ref_tolerance(dtype)
    test.check(LogSumExpFwdOp(dtype=dtype, dim=dim), *test.gen_inputs(), atol=atol, rtol=rtol)


@pytest.mark.gpu
@pytest.mark.parametrize("shape, dim, dtype", [((32, 256), -1, torch.float32),
                                               ((256, 32), 0, torch.float16)])
def test_logsumexp_keepdim(shape, dim, dtype):
    x = torch.randn(*shape, dtype=dtype, device="cuda")
    y = LogSumExpFwdOp(dtype=dtype, dim=dim, keepdim=True)(x)
    ref = _lse_ref(x, dim, keepdim=True)
    assert tuple(y.shape) == ref.shape
    atol, rtol = ref_tolerance(dtype)
    assert_close_np(to_np(y), ref, atol, rtol, "lse keepdim")


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float32, torch.float16])
def test_logsumexp_1d_and_multidim(dtype):
    x = torch.randn(300, dtype=dtype, device="cuda")
    y = LogSumExpFwdOp(dtype=dtype, dim=-1)(x)
    atol, rtol = ref_tolerance(dtype)
    assert y.shape == () and abs(float(y) - float(_lse_ref(x, -1))) <= atol + rtol * abs(float(y))
    x3 = torch.randn(4, 128, 4096, dtype=dtype, device="cuda")
    y3 = LogSumExpFwdOp(dtype=dtype, dim=[0, 2])(x3)
    assert_close_np(to_np(y3), _lse_ref(x3, [0, 2]), atol, rtol, "lse multidim")


@pytest.mark.gpu
@pytest.mark.parametrize("rows", [64, 8192])  # 4 wavefronts per row / 1 per row
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_logsumexp_special_rows(rows, dtype):
    # Finite maxima beyond 2e38 (up to the dtype's largest finite value) must
    # stay finite, as torch.logsumexp keeps them: shift by the max unless it
    # is infinite.
    big = torch.finfo(dtype).max
    x = torch.randn(rows, 4096, device="cuda") * 2
    x[0] = float("-inf")
    x[1, 17] = float("inf")
    x[2, 4000] = float("nan")
    x[3] = 1e30
    x[4, :100] = float("-inf")
    x[5, 7] = 3e38
    x[6] = -3e38
    x[7] = big
    x[8] = -big
    x[9, :2048] = -3e38
    x[9, 2048:] = float("-inf")
    x[10, 5] = float("inf")
    x[10, 6] = float("-inf")
    x[10, 7] = 3e38
    x[11, 3000] = 3e38
    x[11, 3001] = float("nan")
    x = x.to(dtype)
    y = LogSumExpFwdOp(dtype=dtype)(x)
    ref = orc.logsumexp(to_np(x), NAMES[dtype])
    assert np.isfinite(ref[[3, 5, 6, 7, 8, 9]]).all()
    atol, rtol = ref_tolerance(dtype)
    assert_close_np(to_np(y), ref, atol, rtol, "lse special")


@pytest.mark.smoke
def test_logsumexp_eval_roofline_contract():
    with pytest.raises(RuntimeError, match="requires a prior"):
        LogSumExpFwdOp(dtype=torch.float16).eval_roofline()
    with pytest.raises(ValueError, match="Unsupported op_kind"):
        LogSumExpKernel(4, 4, "softmax", torch.float32)


@pytest.mark.gpu
def test_logsumexp_eval_roofline():
    M, N = 64, 256
    op = LogSumExpFwdOp(dim=-1, dtype=torch.float16)
    op(torch.randn(M, N, dtype=torch.float16, device="cuda"))
    assert op.eval_roofline() == (4 * M * N, (M * N + M) * 2)


# -- argmax -----------------------------------------------------------------------------
class ArgmaxTest(ArgmaxWorkload, TestBase):
    def __init__(self, m, n, dtype):
        super().__init__((m, n), dtype)

    def ref_program(self, x):
        return torch.from_numpy(orc.argreduce(to_np(x), -1)).to(x.device)


@pytest.mark.gpu
@pytest.mark.parametrize(
    "m, n, dtype",
    [
        pytest.param(128, 512, torch.float32, marks=pytest.mark.smoke),
        pytest.param(128, 512, torch.float16, marks=pytest.mark.smoke),
        pytest.param(128, 512, torch.bfloat16, marks=pytest.mark.smoke),
        pytest.param(256, 4096, torch.float16, marks=pytest.mark.full),
        pytest.param(256, 4096, torch.bfloat16, marks=pytest.mark.full),
        pytest.param(128, 300, torch.float16, marks=pytest.mark.full),
        pytest.param(128, 300, torch.bfloat16, marks=pytest.mark.full),
        pytest.param(129, 512, torch.float16, marks=pytest.mark.full),
        pytest.param(8192, 4096, torch.float32, marks=pytest.mark.full),
        pytest.param(4, 102400, torch.bfloat16, marks=pytest.mark.full),
    ],
)
def test_argmax_op(m, n, dtype):
    test = ArgmaxTest(m, n, dtype)
    test.check(ArgmaxFwdOp(dtype=dtype, dim=-1), *test.gen_inputs(), compare=_exact_compare)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16])
def test_argmax_ties_nan_and_zeros(dtype):
    x = torch.randint(-3, 4, (512, 777), device="cuda").to(dtype)  # dense ties
    x[0] = float("-inf")
    x[1, [100, 700]] = float("nan")
    x[2] = 0.0
    x[2, :9] = -0.0
    x[3, 776] = float("inf")
    x[4] = float("nan")
    y = ArgmaxFwdOp(dtype=dtype, dim=-1)(x)
    np.testing.assert_array_equal(to_np(y), orc.argreduce(to_np(x), -1))
    np.testing.assert_array_equal(to_np(y), x.cpu().argmax(dim=-1).numpy())


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_argmax_non_contiguous(dtype):
    x = torch.randn(128, 1024, dtype=dtype, device="cuda")[:, :512]
    y = ArgmaxFwdOp(dtype=dtype, dim=-1)(x)
    assert torch.equal(y.cpu(), torch.from_numpy(orc.argreduce(to_np(x.contiguous()), -1)))


@pytest.mark.gpu
@pytest.mark.parametrize(
    "shape, dim, keepdim, dtype",
    [
        ((2, 64, 512), -1, False, torch.float16),
        ((2, 4, 8, 512), -1, False, torch.bfloat16),
        ((512,), -1, False, torch.float32),
        ((4, 8, 256), 0, False, torch.float16),
        ((4, 8, 256), 0, True, torch.float32),
        ((2, 4, 8, 256), 0, True, torch.bfloat16),
        ((128, 512), -1, True, torch.float16),
        ((512, 4, 32), 0, False, torch.float16),
        ((4, 32, 512), 1, False, torch.float16),
        ((4, 32, 512), -1, True, torch.bfloat16),
    ],
)
def test_argmax_dims(shape, dim, keepdim, dtype):
    x = torch.randn(*shape, dtype=dtype, device="cuda")
    y = ArgmaxFwdOp(dtype=dtype, dim=dim, keepdim=keepdim)(x)
    ref = x.cpu().argmax(dim=dim, keepdim=keepdim)
    assert y.shape == ref.shape and y.dtype == torch.int64
    assert torch.equal(y.cpu(), ref)


@pytest.mark.gpu
@pytest.mark.parametrize("shape, dtype", [((16, 64), torch.float16), ((16, 64), torch.bfloat16),
                                          ((16, 64), torch.float32), ((512,), torch.float16),
                                          ((4, 8, 32), torch.float16), ((2, 4, 8, 16), torch.float16),
                                          ((10, 30), torch.float16)])
def test_argmax_dim_none(shape, dtype):
    x = torch.randn(*shape, dtype=dtype, device="cuda")
    ref = torch.argmax(x.cpu())
    y = ArgmaxFwdOp(dtype=dtype, dim=None)(x)
    assert y.dtype == torch.int64 and y.shape == ref.shape and torch.equal(y.cpu(), ref)
    yk = ArgmaxFwdOp(dtype=dtype, dim=None, keepdim=True)(x)
    assert yk.shape == tuple(1 for _ in shape) and torch.equal(yk.reshape(()).cpu(), ref)


@pytest.mark.smoke
@pytest.mark.parametrize("dim", [[0, 1], (0, 1)])
def test_argmax_rejects_multidim(dim):
    with pytest.raises((TypeError, ValueError)):
        ArgmaxFwdOp(dtype=torch.float16, dim=dim)


@pytest.mark.smoke
def test_argreduce_kernel_contract():
    with pytest.raises(ValueError, match="Unsupported op_kind"):
        ArgreduceKernel(4, 4, "argsort", torch.float32)
    with pytest.raises(ValueError, match="empty"):
        ArgreduceKernel(4, 0, "argmax", torch.float32)


@pytest.mark.gpu
@pytest.mark.parametrize("M, N, dtype", [
    (1, 600000, torch.float32),    # several workgroups per row, merged
    (128, 131073, torch.float16),  # the most rows that split, odd length
    (129, 131073, torch.float16),  # one 16-wavefront workgroup per row
    (512, 16384, torch.float32),   # sixteen wavefronts per row
    (513, 16381, torch.bfloat16),  # four
    (3072, 1027, torch.bfloat16),  # one
    (5, 3, torch.float16),         # short rows: elements, 4 lanes each
    (1001, 13, torch.bfloat16),    # 16
    (70, 64, torch.float32),       # packs, 16 lanes
    (9, 17, torch.float16),        # ragged packs, 16 lanes
    (600, 131, torch.float32),     # 32
    (77, 519, torch.float16),      # 64 packs and both edges
    (5000, 512, torch.float16),    # packs, 64 lanes
    (6, 521, torch.bfloat16),      # the shortest ragged row past them
])
def test_row_split_and_ragged_rows(M, N, dtype):
    # extremes at the row's first and last elements and around the first and
    # last aligned pack: each must be seen exactly once by the plan
    x = torch.randn(M, N, device="cuda").to(dtype)
    rows = torch.arange(M, device="cuda")
    where = torch.tensor([0, N - 1, min(7, N - 1), max(0, N - 8), N // 2], device="cuda")
    x[rows, where[rows % 5]] = 30.0
    x[0, N // 3] = float("nan")
    got = ArgmaxFwdOp(dtype=dtype, dim=-1)(x)
    assert torch.equal(got.cpu(), torch.argmax(x.cpu(), dim=-1))
    # fp32 sums of N positive terms: N eps relative in the sum, far below
    # atol on its logarithm
    x[0, N // 3] = 0.0
    y = LogSumExpFwdOp(dtype=dtype)(x)
    atol, rtol = ref_tolerance(dtype)
    assert_close_np(to_np(y), torch.logsumexp(x.double(), -1).cpu().numpy(), atol, rtol, "lse")


# -- reductions over other dims, read as they lie -----------------------------------------
def test_strided_form_matches_the_general_path():
    # every dim set of shapes with size-1 dims: the view reduces to what the
    # permuted copy reduces to; views that are not contiguous are refused
    import itertools

    from tileops.ops._multidim import flatten_for_multidim, strided_form

    seen = {False: 0, True: 0}
    for shape in ((5, 64), (3, 4, 70), (2, 3, 4, 66), (3, 1, 64), (1, 7, 64, 1), (2, 65, 1, 3),
                  (64, 2, 3, 64)):
        x = torch.randn(shape, dtype=torch.float64)
        for k in range(1, len(shape) + 1):
            for dims in itertools.combinations(range(len(shape)), k):
                form = strided_form(x, list(dims))
                if form is None:
                    continue
                outer, n, inner, ends = form
                seen[ends] += 1
                v = x.view(outer, n, inner)
                y = torch.logsumexp(v, (0, 2) if ends else (1,)).reshape(-1)
                flat, _, _ = flatten_for_multidim(x, list(dims))
                ref = torch.logsumexp(flat, -1).reshape(-1)
                torch.testing.assert_close(y, ref, rtol=1e-12, atol=1e-12)
                if not ends and len(dims) == 1:
                    assert torch.equal(v.argmax(1).reshape(-1), flat.argmax(-1).reshape(-1))
    assert seen[False] >= 8 and seen[True] >= 3
    x = torch.randn(4, 128, 64)
    assert strided_form(x.transpose(0, 1), [0]) is None
    assert strided_form(x[:, ::2], [0]) is None
    assert strided_form(x[:, :, :63].contiguous(), [1]) is None  # too few columns
    assert strided_form(torch.empty(0, 4, 64), [0]) is None
    assert strided_form(torch.empty(20000, 2, 64), [0, 2]) is None  # too many partials


@pytest.mark.gpu
@pytest.mark.parametrize("shape, dim, dtype", [
    ((4, 128, 4096), 0, torch.float16),    # 256 threads across the columns, 4 rows
    ((3, 5, 67), 1, torch.bfloat16),       # one column per thread, ragged tile
    ((2, 33, 200), 1, torch.float32),      # 50 packs, 16 across
    ((2, 1000, 1024), 1, torch.float16),   # 16 row groups per column
    ((9, 40, 70, 64), 1, torch.float32),   # 64 across, several tiles
    ((20000, 64), 0, torch.float32),       # split over workgroups
    ((20001, 65), 0, torch.bfloat16),      # split, one column per thread
    ((1, 1, 64), 1, torch.float16),        # one row
])
def test_reductions_over_an_inner_dim(shape, dim, dtype):
    x = torch.randn(shape, device="cuda").to(dtype)
    n = shape[dim]
    x.select(dim, n - 1)[..., ::3] = 9.0  # extremes in the last and first rows
    x.select(dim, 0)[..., 1::3] = 9.0
    x.view(-1)[5] = float("nan")
    assert torch.equal(ArgmaxFwdOp(dtype=dtype, dim=dim)(x).cpu(), torch.argmax(x.cpu(), dim=dim))
    x.view(-1)[5] = float("-inf")
    y = LogSumExpFwdOp(dtype=dtype, dim=dim, keepdim=True)(x)
    atol, rtol = ref_tolerance(dtype)
    ref = torch.logsumexp(x.double(), dim, keepdim=True).cpu().numpy()
    assert_close_np(to_np(y), ref, atol, rtol, "lse over an inner dim")
    # a contiguous view whose base is off the 16-byte grid
    off = torch.empty(x.numel() + 1, device="cuda", dtype=dtype)[1:].view(shape).copy_(x)
    assert torch.equal(ArgmaxFwdOp(dtype=dtype, dim=dim)(off), ArgmaxFwdOp(dtype=dtype, dim=dim)(x))


@pytest.mark.gpu
@pytest.mark.parametrize("shape, dims, dtype", [
    ((4, 128, 4096), [0, 2], torch.float16),  # rows of several wavefronts
    ((33, 3, 100), [0, 2], torch.float32),    # short rows
    ((70, 2, 203), [0, 2], torch.bfloat16),   # ragged rows
    ((2, 1, 600000), [0, 2], torch.float32),  # rows split over workgroups too
    ((6, 5, 4, 64), [0, 1, 3], torch.float32),
    ((6, 5, 4, 64), [0, 1], torch.float16),
])
def test_logsumexp_over_several_dims(shape, dims, dtype):
    x = (torch.randn(shape, device="cuda") * 2).to(dtype)
    y = LogSumExpFwdOp(dtype=dtype, dim=dims)(x)
    atol, rtol = ref_tolerance(dtype)
    assert_close_np(to_np(y), torch.logsumexp(x.double(), dims).cpu().numpy(), atol, rtol, "lse")


def test_strided_form_leaves_large_sizes_to_the_general_path():
    # a size past the entry point's 31 bits, wherever it stands; the largest
    # sizes below it are taken
    from tileops.ops._multidim import strided_form

    def form(shape, dims):
        return strided_form(torch.empty(shape, device="meta"), dims)

    big = 2**31
    for shape, dims in (((2, big), [0]), ((big, 2, 64), [1]), ((2, big, 64), [1]),
                        ((2, 3, big), [0, 1]), ((2, big, 64), [0, 2]), ((2, 3, big // 2), [0, 2])):
        assert form(shape, dims) is None, (shape, dims)
    assert form((2, big - 1), [0]) == (1, 2, big - 1, False)
    assert form((big - 1, 4, 64), [1]) == (big - 1, 4, 64, False)
    assert form((2, big - 1, 64), [0, 2]) == (2, big - 1, 64, True)
    assert form((2, 3, big // 2 - 1), [0, 2]) == (2, 3, big // 2 - 1, True)
    # many small slices are copied: from 16384 on, below 64 packs of 16 bytes
    assert strided_form(torch.empty((16384, 3, 84), device="meta"), [1]) is None
    assert form((16384, 4, 64), [1]) == (16384, 4, 64, False)
    assert form((16383, 3, 84), [1]) == (16383, 3, 84, False)
    half = torch.empty((16384, 4, 64), device="meta", dtype=torch.float16)
    assert strided_form(half, [1]) is None


def _windows(n):
    """The ends, and around multiples of 2^24 workgroups of 4 to 64 rows."""
    at = [0, n - 100] + [k for e in (24, 26, 28, 30) for k in (2**e - 50,) if k + 100 < n]
    return [slice(i, i + 100) for i in at]


@pytest.mark.gpu
@pytest.mark.parametrize("shape, dim, dtype", [
    ((2**28 + 40, 5), -1, torch.float16),     # short rows, sixteen to a workgroup
    ((2, 2**31 + 64), 0, torch.bfloat16),     # copied, short rows past 2^31
    ((2**24 + 3, 8, 64), 1, torch.bfloat16),  # a column workgroup per outer slice
    ((2**24 + 3, 2, 64), 1, torch.bfloat16),  # copied
    ((2, 2**26 + 9, 64), [0, 2], torch.float16),  # merged from partials
])
def test_reductions_of_more_rows_than_one_launch_holds(shape, dim, dtype):
    # 2^32 threads and more: each launch goes in slices
    if torch.cuda.mem_get_info()[0] < 40 << 30:
        pytest.skip("needs 40 GB of device memory")
    x = torch.empty(shape, device="cuda", dtype=dtype).normal_()
    y = LogSumExpFwdOp(dtype=dtype, dim=dim)(x)
    i = ArgmaxFwdOp(dtype=dtype, dim=dim)(x) if isinstance(dim, int) else None
    kept = 1 if dim == 0 or not isinstance(dim, int) else 0
    atol, rtol = ref_tolerance(dtype)
    for w in _windows(x.shape[kept]):
        part = x[:, w] if kept == 1 else x[w]
        ref = torch.logsumexp(part.double(), dim).cpu().numpy()
        assert_close_np(to_np(y[w]), ref, atol, rtol, f"lse {w}")
        if i is not None:
            assert torch.equal(i[w].cpu(), torch.argmax(part.cpu(), dim=dim))


# -- the C functions with and without scratch ----------------------------------------------
def _reduce(op, x, room):
    """tileops_reduce_fwd of the rows of x with ``room(need)`` bytes of scratch."""
    lib, (M, N) = _native.lib(), x.shape
    code = _native.dtype_code(x.dtype)
    need = lib.tileops_reduce_workspace_bytes(M, N, code)
    room = room(need)
    ws = torch.empty(max(room, 1), dtype=torch.uint8, device=x.device)
    y = torch.empty(M, dtype=x.dtype if op == _native.LOGSUMEXP else torch.int64, device=x.device)
    _native.check(lib.tileops_reduce_fwd(op, x.data_ptr(), y.data_ptr(), M, N, code,
                                         ws.data_ptr() if room else None, room,
                                         _native.stream_of(x)), "tileops_reduce_fwd")
    return y, need


@pytest.mark.gpu
@pytest.mark.parametrize("M, N, dtype", [
    (1, 600000, torch.float32),
    (4, 131072, torch.bfloat16),   # the shortest rows that split
    (128, 131073, torch.float16),  # the most rows, ragged
])
def test_rows_with_and_without_scratch(M, N, dtype):
    x = torch.randn(M, N, device="cuda").to(dtype)
    x[:, N // 3] = x[:, N - 2] = 30.0  # a tie: the first wins
    atol, rtol = ref_tolerance(dtype)
    ref = torch.logsumexp(x.double(), -1).cpu().numpy()
    lib = _native.lib()
    code = _native.dtype_code(dtype)
    for room in (lambda need: 0, lambda need: need - 1, lambda need: need):
        i, need = _reduce(_native.ARGMAX, x, room)
        assert need > 0 and torch.equal(i.cpu(), torch.full((M,), N // 3))
        assert torch.equal(_reduce(_native.ARGMIN, -x, room)[0], i)
        assert_close_np(to_np(_reduce(_native.LOGSUMEXP, x, room)[0]), ref, atol, rtol, "lse")
    i = torch.empty(M, dtype=torch.int64, device="cuda")
    y = torch.empty(M, dtype=dtype, device="cuda")
    s = _native.stream_of(x)
    assert lib.tileops_argreduce_fwd(x.data_ptr(), i.data_ptr(), M, N, code, 0, s) == 0
    assert lib.tileops_logsumexp_fwd(x.data_ptr(), y.data_ptr(), M, N, code, s) == 0
    assert torch.equal(i.cpu(), torch.full((M,), N // 3))
    assert_close_np(to_np(y), ref, atol, rtol, "lse without scratch")


@pytest.mark.smoke
def test_reduce_entry_points_reject_bad_scratch():
    lib, p = _native.lib(), 4096  # non-null host values: refused before any launch
    need = lib.tileops_reduce_axis_workspace_bytes(1, 1, 20000, 64, 0, 0)  # columns split
    assert need > 0
    axis = lib.tileops_reduce_axis_fwd
    assert axis(1, p, p, 1, 20000, 64, 0, 0, None, 0, None) == -4
    assert axis(1, p, p, 1, 20000, 64, 0, 0, None, need, None) == -4
    assert axis(1, p, p, 1, 20000, 64, 0, 0, p, need - 1, None) == -4
    assert axis(1, p, p, 1, 20000, 64, 0, 0, p + 4, need, None) == -1
    assert axis(0, p, p, 8, 4, 64, 1, 0, None, 0, None) == -4  # both ends: merged from partials
    assert lib.tileops_reduce_axis_workspace_bytes(0, 8, 4, 64, 1, 0) == 8 * 4 * 8
    assert axis(1, p, p, 8, 4, 64, 1, 0, p, 1 << 20, None) == -1  # no index over both ends
    assert axis(3, p, p, 8, 4, 64, 0, 0, None, 0, None) == -1
    assert axis(0, p, p, 8, 0, 64, 0, 0, None, 0, None) == -2
    assert axis(0, p, p, 8, 4, 2**31, 0, 0, None, 0, None) == -2
    assert axis(0, None, p, 8, 4, 64, 0, 0, None, 0, None) == -3
    rows = lib.tileops_reduce_fwd
    assert rows(0, p, p, 4, 131072, 2, p + 8, 1 << 20, None) == -1
    assert rows(3, p, p, 4, 64, 2, None, 0, None) == -1
    assert rows(0, p, p, 4, 0, 2, None, 0, None) == -2
    assert rows(0, None, None, 0, 64, 2, None, 0, None) == 0
    # which rows split: at most 128, of 256 chunks of 64 packs and more
    ask = lib.tileops_reduce_workspace_bytes
    assert ask(4, 131072, 2) > 0 and ask(128, 131072, 2) > 0
    assert ask(129, 131072, 2) == 0 and ask(4, 130560, 2) == 0


@pytest.mark.gpu
@pytest.mark.parametrize("shape, dim, dtype", [
    ((6, 131080), 1, torch.bfloat16),    # rows split over workgroups, merged
    ((6, 600001), 1, torch.float32),     # ragged
    ((6, 4, 128), 1, torch.float16),     # columns, few rows
    ((2, 1000, 128), 1, torch.bfloat16),  # 16 row groups per column
    ((20000, 128), 0, torch.float32),    # columns split, merged
    ((20001, 65), 0, torch.float16),
    ((70, 6, 203), [0, 2], torch.bfloat16),  # partials of short ragged rows
    ((2, 6, 600000), [0, 2], torch.float32),  # partials of split rows
])
def test_special_values_in_every_plan(shape, dim, dtype):
    # one output of each kind: all -inf, one +inf, a NaN, all the type's lowest
    # value, the lowest with one zero, the largest value (kept finite)
    x = torch.randn(shape, device="cuda").to(dtype)
    dims = [dim] if isinstance(dim, int) else dim
    kept = [d for d in range(len(shape)) if d not in dims][-1]
    info = torch.finfo(dtype)

    def put(i, all_, last=None):
        sel = x.select(kept, i)
        if all_ is not None:
            sel.fill_(all_)
        if last is not None:
            sel.movedim([d - (d > kept) for d in dims], list(range(-len(dims), 0)))[
                (...,) + (-1,) * len(dims)] = last

    for i, (all_, last) in enumerate([(float("-inf"), None), (None, float("inf")),
                                      (None, float("nan")), (info.min, None), (info.min, 0.0),
                                      (0.0, info.max)]):
        put(i, all_, last)
    y = to_np(LogSumExpFwdOp(dtype=dtype, dim=dim)(x))
    ref = torch.logsumexp(x.double(), dim).to(dtype).float().cpu().numpy()
    atol, rtol = ref_tolerance(dtype)
    assert_close_np(y, ref, atol, rtol, "lse")
    if isinstance(dim, int):
        assert torch.equal(ArgmaxFwdOp(dtype=dtype, dim=dim)(x).cpu(), torch.argmax(x.cpu(), dim))
