"""Which calls may skip the torch.library custom op: plain eager ones only."""

import pytest
import torch
from torch._subclasses.fake_tensor import FakeTensorMode
from torch.utils._python_dispatch import TorchDispatchMode

from tileops import _native


def _seen(*tensors):
    """What ``eager`` says from inside the context the caller is in."""
    return _native.eager(*tensors)


def test_plain_calls():
    x = torch.ones(3)
    assert _seen(x, torch.nn.Parameter(x, requires_grad=False))
    y = torch.ones(3, requires_grad=True)
    assert not _seen(x, y)
    with torch.no_grad():
        assert _seen(x, y)
    with torch.inference_mode():
        assert _seen(x)


@pytest.mark.parametrize("make", [
    lambda: torch.full((1, 1), 2 + 3j).conj().imag,  # negative bit, contiguous
    lambda: torch._neg_view(torch.ones(4, 64)),
    lambda: torch._efficientzerotensor((3,)),
], ids=["conj_imag", "neg_view", "zerotensor"])
def test_lazy_tensors_take_the_custom_op(make):
    # the storage does not hold the values: the dispatcher materialises them
    # for the custom op, a raw pointer would be read as it lies
    x = make()
    assert x.is_contiguous()
    assert not _seen(x) and not _seen(torch.ones(3), x)
    got = []

    @torch.library.custom_op("tileops_test::eager_probe", mutates_args=())
    def probe(t: torch.Tensor) -> torch.Tensor:
        got.append((t.is_neg(), t._is_zerotensor()))
        return t.clone()

    assert torch.equal(probe(x), x + 0) and got == [(False, False)]


@pytest.mark.gpu
def test_negative_views_on_the_gpu():
    from tileops.ops.reduction import ArgmaxFwdOp, LogSumExpFwdOp

    x = torch.randn(5, 64, generator=torch.Generator().manual_seed(3)).cuda()
    neg = torch._neg_view(x)
    assert torch.equal(LogSumExpFwdOp(dtype=torch.float32)(neg),
                       LogSumExpFwdOp(dtype=torch.float32)(-x))
    assert torch.equal(ArgmaxFwdOp(dtype=torch.float32, dim=-1)(neg), torch.argmin(x, dim=-1))


class _Sub(torch.Tensor):
    pass


class _Mode(TorchDispatchMode):
    def __torch_dispatch__(self, func, types, args=(), kwargs=None):
        return func(*args, **(kwargs or {}))


class _FnMode(torch.overrides.TorchFunctionMode):
    def __torch_function__(self, func, types, args=(), kwargs=None):
        return func(*args, **(kwargs or {}))


@pytest.mark.parametrize("mode", [_Mode, _FnMode, FakeTensorMode, torch.autograd.forward_ad.dual_level])
def test_modes_take_the_custom_op(mode):
    x = torch.ones(3)
    with mode():
        assert not _seen(x)
    assert _seen(x)


def test_subclasses_transforms_and_tracing_take_the_custom_op():
    assert not _seen(torch.ones(3).as_subclass(_Sub))
    got = []

    def probe(x):
        got.append(_seen(x))
        return x * 2

    torch.vmap(probe)(torch.ones(2, 3))
    torch.func.jvp(probe, (torch.ones(3),), (torch.ones(3),))
    torch.jit.trace(probe, torch.ones(3), check_trace=False)
    torch.compile(probe, backend="eager", fullgraph=False)(torch.ones(3))
    torch._dynamo.reset()
    assert got == [False] * len(got) and len(got) >= 3
