"""Which calls of a linear may go to the hand-written products (CPU): plain
values only, and modules whose hooks nobody would miss."""

from __future__ import annotations

import pytest
import torch
from torch.autograd import forward_ad

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
