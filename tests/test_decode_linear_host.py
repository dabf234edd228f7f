"""Routing of DecodeLinear on the CPU: the kernel is stood in for by torch's own product, so that only the question who is asked remains."""

import pytest
import torch
import torch.nn as nn
import torch.nn.functional as F
from torch.nn.modules import module as torch_module

from easy_to_hard_amd import feed_forward, seq_ops
from easy_to_hard_amd.feed_forward import ExpertMixture, SquaredReluFF
from easy_to_hard_amd.linear import DecodeLinear, fusable


@pytest.fixture
def streamed(monkeypatch):
    """every linear streams; returns the weights that the joined product + activation was launched with"""
    joined = []

    def linear(x, weight, act=seq_ops.ACT_NONE, cap=0.0):
        y = F.linear(x, weight)
        if act == seq_ops.ACT_SQUARE_RELU:
            joined.append(weight)
            y = F.relu(y).square()
        return y

    monkeypatch.setattr(seq_ops, "linear_streams", lambda x, weight: True)
    monkeypatch.setattr(seq_ops, "linear", linear)
    monkeypatch.setattr(seq_ops, "square_relu_", lambda x: F.relu(x).square())
    return joined


def _watchers():
    def own_forward(lin, seen):
        inner = lin.forward
        lin.forward = lambda x: (seen.append(1), inner(x))[1]

    def globally(register):
        def put(lin, seen):
            return register(lambda module, *args: seen.append(1) if module is lin else None)

        return put

    return {
        "forward of the instance": own_forward,
        "forward hook": lambda lin, seen: lin.register_forward_hook(lambda *a: seen.append(1)),
        "forward pre-hook": lambda lin, seen: lin.register_forward_pre_hook(lambda *a: seen.append(1)),
        "global forward hook": globally(torch_module.register_module_forward_hook),
        "global forward pre-hook": globally(torch_module.register_module_forward_pre_hook),
    }


@pytest.mark.parametrize("how", _watchers())
def test_a_watched_linear_is_called_as_a_module(streamed, how):
    ff = SquaredReluFF(16, 24)
    x = torch.randn(3, 16)
    want = F.linear(F.relu(F.linear(x, ff.up.weight)).square(), ff.down.weight)
    assert torch.equal(ff(x), want) and len(streamed) == 1
    seen = []
    handle = _watchers()[how](ff.up, seen)
    try:
        assert torch.equal(ff(x), want)
        assert len(seen) == 1 and len(streamed) == 1
    finally:
        if handle is not None:
            handle.remove()


@pytest.mark.parametrize("register", [torch_module.register_module_full_backward_hook, torch_module.register_module_full_backward_pre_hook])
def test_global_backward_hooks_keep_the_module_call(streamed, register):
    lin = DecodeLinear(16, 24, bias=False)
    assert fusable(lin, torch.randn(2, 16))
    handle = register(lambda *a: None)
    try:
        assert not fusable(lin, torch.randn(2, 16))
    finally:
        handle.remove()


@pytest.mark.parametrize("which", ["up", "down"])
@pytest.mark.parametrize("how", _watchers())
def test_a_watched_shared_expert_is_called_as_a_module(streamed, monkeypatch, which, how):
    """the shared expert runs inside the experts' launches only while nobody watches its linears"""
    taken = []

    def experts(h, chosen, up, down, shared_up=None, shared_down=None):
        taken.append(shared_up is not None)
        return h, (None if shared_up is None else F.linear(F.relu(F.linear(h, shared_up)).square(), shared_down))

    monkeypatch.setattr(feed_forward.seq_ops, "route", lambda h, *a: (None, None))
    monkeypatch.setattr(feed_forward.seq_ops, "experts", experts)
    mix = ExpertMixture(16, 4, 2, 8, 24)
    x = torch.randn(3, 16)
    shared = mix(x)[0]
    assert taken == [True]
    seen = []
    handle = _watchers()[how](getattr(mix.shared, which), seen)
    try:
        assert torch.equal(mix(x)[0], shared)
        assert seen == [1] and taken == [True, False]
    finally:
        if handle is not None:
            handle.remove()


def test_plain_linears_of_a_replaced_module_are_left_alone(streamed):
    ff = SquaredReluFF(16, 24)
    ff.up = nn.Linear(16, 24, bias=False)
    x = torch.randn(3, 16)
    assert torch.equal(ff(x), F.linear(F.relu(F.linear(x, ff.up.weight)).square(), ff.down.weight)) and not streamed
