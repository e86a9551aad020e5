"""Which calls of a linear may go to the hand-written products (CPU): plain
values only, and modules whose hooks nobody would miss."""

from __future__ import annotations

import copy
import ctypes
import pickle

import pytest
import torch
from torch._subclasses.fake_tensor import FakeTensorMode
from torch.autograd import forward_ad
from torch.fx.experimental.proxy_tensor import make_fx
from torch.overrides import TorchFunctionMode
from torch.utils._python_dispatch import _disable_current_modes
from torch.utils.flop_counter import FlopCounterMode

from ppu_amd import integration


def test_values_only():
    x, w = torch.randn(1, 8), torch.randn(4, 8)
    assert integration._values_only(x, w)
    wg = w.clone().requires_grad_()
    assert not integration._values_only(x, wg)
    with torch.no_grad():
        assert integration._values_only(x, wg)
    with forward_ad.dual_level():
        assert not integration._values_only(forward_ad.make_dual(x, torch.ones_like(x)), w)
    seen = []
    torch.vmap(lambda row: seen.append(integration._values_only(row, w)) or row)(x)
    assert seen == [False]


HOOKS = ["register_forward_hook", "register_forward_pre_hook", "register_full_backward_hook",
         "register_full_backward_pre_hook"]


@pytest.mark.parametrize("name", HOOKS)
def test_hooked_linear_is_called(name):
    linear = torch.nn.Linear(8, 4)
    calls = []
    getattr(linear, name)(lambda *args: calls.append(name))
    integration._bias_module(linear, torch.randn(3, 8, requires_grad=True)).sum().backward()
    assert calls == [name]


def test_global_hook_sees_the_linear():
    calls = []
    handle = torch.nn.modules.module.register_module_forward_hook(lambda *args: calls.append(1))
    try:
        integration._bias_module(torch.nn.Linear(8, 4), torch.randn(3, 8))
    finally:
        handle.remove()
    assert calls == [1]


@pytest.fixture
def head(monkeypatch):
    """A language model head on the CPU whose fast path is taken as on the GPU
    and, as there, writes its output through its address alone."""
    def by_address(x, w):
        y = torch.empty(*x.shape[:-1], w.shape[0], dtype=x.dtype)
        with _disable_current_modes():
            value = torch.nn.functional.linear(x.detach().clone(), w.detach().clone())
        ctypes.memmove(y.data_ptr(), value.data_ptr(), value.numel() * value.element_size())
        return y

    linear = torch.nn.Linear(8, 4, bias=False).to(torch.bfloat16).requires_grad_(False)
    monkeypatch.setattr(integration, "_gpu_bf16", lambda t: t.dtype == torch.bfloat16)
    monkeypatch.setattr(integration.K, "linear", by_address)
    integration._take_over(linear, integration._lm_head_fast(linear))
    return linear


def _row(seed):
    return torch.randn(1, 8, generator=torch.Generator().manual_seed(seed)).to(torch.bfloat16)


def test_plain_call_takes_the_fast_path(head, monkeypatch):
    taken = []
    monkeypatch.setattr(integration.K, "linear", lambda x, w: taken.append(1) or x[:, :4])
    with torch.device("cpu"):  # a default device is not a tracer
        head(_row(1))
    assert taken == [1]


@pytest.mark.parametrize("trace", [
    lambda f, x: torch.jit.trace(f, x, check_trace=False), lambda f, x: make_fx(f)(x),
    lambda f, x: make_fx(f, pre_dispatch=True)(x)])
def test_traced_head_computes_its_logits(head, trace):
    traced = trace(lambda x: head(x), _row(1))
    x = _row(2)
    assert torch.equal(traced(x), torch.nn.functional.linear(x, head.weight))


def test_modes_see_the_product(head):
    with FlopCounterMode(display=False) as flops:
        head(_row(1))
    assert flops.get_total_flops() == 2 * 8 * 4
    with FakeTensorMode() as mode:
        x, w = mode.from_tensor(_row(1)), mode.from_tensor(head.weight)
        assert not integration._values_only(x, w) and not integration._values_only(x)
    with FakeTensorMode(allow_non_fake_inputs=True):
        assert not integration._values_only(_row(1))
    seen = []

    class Mode(TorchFunctionMode):
        def __torch_function__(self, func, types, args=(), kwargs=None):
            seen.append(func)
            return func(*args, **(kwargs or {}))

    with Mode():
        head(_row(1))
    assert torch.nn.functional.linear in seen or torch._C._nn.linear in seen


class _Packed(torch.Tensor):
    """A wrapper subclass as quantised weights are: it says cuda and bf16, has
    no storage and multiplies in its own way."""

    @staticmethod
    def __new__(cls, shape):
        return torch.Tensor._make_wrapper_subclass(cls, shape, dtype=torch.bfloat16, device="cuda")

    @classmethod
    def __torch_function__(cls, func, types, args=(), kwargs=None):
        if func is torch.nn.functional.linear:
            return "its own product"
        with torch._C.DisableTorchFunctionSubclass():
            return func(*args, **(kwargs or {}))

    @classmethod
    def __torch_dispatch__(cls, func, types, args=(), kwargs=None):
        if func is torch.ops.aten.detach.default:
            return _Packed(args[0].shape)
        raise NotImplementedError(func)


def test_weight_subclass_keeps_its_product(head):
    head.weight = torch.nn.Parameter(_Packed((4, 8)), requires_grad=False)
    assert head(_row(1)) == "its own product"
    x, w, b = _row(1), torch.randn(4, 64).to(torch.bfloat16), torch.randn(4).to(torch.bfloat16)
    assert integration._values_only(x, w, torch.nn.Parameter(b, requires_grad=False))
    assert not integration._values_only(x, head.weight, b) and not integration._values_only(_Packed((1, 8)), w, b)
    assert integration._bias_linear(x, head.weight, b) == "its own product"


def test_sparse_and_nested_operands_keep_the_module(head):
    rows = [_row(1).float(), _row(2).float()]
    with torch.no_grad():
        assert not integration._values_only(torch.nested.nested_tensor(rows))
        dense = head.weight.float()
        assert not integration._values_only(dense.to_sparse_csr()) and not integration._values_only(dense.to_sparse())
        nested = torch.nested.nested_tensor([r.to(torch.bfloat16) for r in rows])
        assert head(nested).is_nested


def _installed_head(fused):
    off = dict.fromkeys(("delta", "rms_norm", "residual_norm", "swiglu", "attention", "vision", "lm_head_screen"),
                        False)
    model = torch.nn.Module()
    model.model = torch.nn.Module()
    model.model.layers = torch.nn.ModuleList()
    model.lm_head = torch.nn.Linear(2048, 4, bias=False)
    integration.install(model.eval(), integration.FusionConfig(**off, fused_decode=fused), [])
    return model.lm_head


def test_head_is_taken_over_with_fused_decode_only():
    """Every fusion off leaves the head as it was."""
    assert "forward" in _installed_head(True).__dict__
    assert "forward" not in _installed_head(False).__dict__


@pytest.mark.parametrize("twin", [copy.deepcopy, lambda head: pickle.loads(pickle.dumps(head))])
def test_copied_head_uses_its_own_weight(twin):
    head = _installed_head(True)
    other, x = twin(head), torch.ones(1, 2048)
    with torch.no_grad():
        other.weight.fill_(2.0)
        assert other(x).eq(4096).all() and not head(x).eq(4096).any()
    other(x).sum().backward()
    assert other.weight.grad is not None and head.weight.grad is None


@pytest.mark.parametrize("n,k", [(0, 64), (4, 0)])
def test_empty_linear_keeps_the_library(monkeypatch, n, k):
    """No columns or no terms, or one bias for all columns: F.linear answers,
    the GEMM's entry refuses."""
    def refused(*args, **kwargs):
        raise RuntimeError

    monkeypatch.setattr(integration, "_gpu_bf16", lambda t: t.dtype == torch.bfloat16)
    monkeypatch.setattr(integration.K, "gemm_bias", refused)
    monkeypatch.setattr(integration.K, "linear", refused)
    x, w, b = (torch.ones(*s, dtype=torch.bfloat16) for s in ((3, k), (n, k), (n,)))
    assert torch.equal(integration._bias_linear(x, w, b), torch.ones(3, n, dtype=torch.bfloat16))
    one = torch.ones(1, dtype=torch.bfloat16)  # a bias for every column
    assert integration._bias_linear(torch.ones(3, 64, dtype=torch.bfloat16), w.new_ones(4, 64), one).eq(65).all()
    head = torch.nn.Linear(k, n, bias=False).to(torch.bfloat16).requires_grad_(False)
    integration._take_over(head, integration._lm_head_fast(head))
    assert head(x[:1]).shape == (1, n)


@pytest.mark.parametrize("m,n,k,ours", [(784, 4352, 1152, True), (1296, 4352, 1152, True), (1444, 4352, 1152, False),
                                        (1800, 1152, 4352, False), (4096, 1152, 1152, True),
                                        (306, 4608, 4608, True), (400, 4608, 4608, False)])
def test_linear_route_by_work(monkeypatch, m, n, k, ours):
    """The hand-written product where it is the faster one, the library's from
    6.5e9 multiply-adds up."""
    taken = []
    monkeypatch.setattr(integration, "_gpu_bf16", lambda t: t.dtype == torch.bfloat16)
    monkeypatch.setattr(integration.K, "gemm_bias", lambda x, w, b, gelu: taken.append(True))
    monkeypatch.setattr(torch.nn.functional, "linear", lambda x, w, b: taken.append(False))
    integration._bias_linear(*(torch.empty(*s, dtype=torch.bfloat16) for s in ((m, k), (n, k), (n,))))
    assert taken == [ours]
