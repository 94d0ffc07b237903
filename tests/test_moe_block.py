"""MoEFeedForwardBlock calls its submodules as modules wherever somebody could tell: replaced, wrapped or
compiled `forward`s and hooks.  On the CPU, where the kernels cannot run: the parts that would launch them
are the ones replaced."""
import pytest
import torch
from torch import nn

from piper_amd import functional as F_
from piper_amd import moe as M

X = torch.randn(2, 3, 16)


def _block():
    torch.manual_seed(0)
    blk = M.MoEFeedForwardBlock(M.MoEArgs(num_experts=4, top_k=2), dim=16, hidden_dim=8, dtype=torch.float32)
    blk.moe.init_weights()
    return blk


def _norm_double(self, x):
    return 2 * x


def _moe_add(self, x, residual=None):
    return 3 * x + residual


WANT = 3 * (2 * X) + X


def test_forward_replaced_on_the_instances():
    blk = _block()
    blk.ffn_norm.forward = lambda x: 2 * x
    blk.moe.forward = lambda x, residual=None: 3 * x + residual
    assert torch.equal(blk(X), WANT)


@pytest.mark.parametrize("part", ["ffn_norm", "moe"])
def test_forward_replaced_on_one_instance(part):
    blk = _block()
    getattr(blk, part).forward = lambda x, residual=None: x
    assert not blk._one_node()


def test_forward_patched_on_the_classes(monkeypatch):
    monkeypatch.setattr(M.RMSNorm, "forward", _norm_double)
    monkeypatch.setattr(M.AnnotatedMoE, "forward", _moe_add)
    assert torch.equal(_block()(X), WANT)


@pytest.mark.parametrize("attr", ["_call_impl", "__call__"])
def test_module_call_patched(monkeypatch, attr):
    """Tracers and profilers put a function of their own in place of nn.Module's call."""
    blk = _block()
    assert blk._one_node()
    original = getattr(nn.Module, attr)
    monkeypatch.setattr(nn.Module, attr, lambda self, *a, **kw: original(self, *a, **kw))
    assert not blk._one_node()


def test_compiled_submodule():
    blk = _block()
    blk.ffn_norm.forward = lambda x: 2 * x
    blk.moe.forward = lambda x, residual=None: 3 * x + residual
    blk2 = _block()
    calls = []

    def backend(gm, example_inputs):
        calls.append(gm)
        return gm.forward

    blk2.moe.compile(backend=backend)
    assert not blk2._one_node()
    blk.moe.compile(backend=backend)
    assert torch.equal(blk(X), WANT) and calls


@pytest.mark.parametrize("register", ["register_module_forward_hook", "register_module_forward_pre_hook",
                                      "register_module_full_backward_hook", "register_module_full_backward_pre_hook"])
def test_global_module_hooks(register):
    blk = _block()
    assert blk._one_node()
    handle = getattr(nn.modules.module, register)(lambda *a: None)
    try:
        assert not blk._one_node()
    finally:
        handle.remove()
    assert blk._one_node()


@pytest.mark.parametrize("register", ["register_forward_hook", "register_forward_pre_hook", "register_full_backward_hook",
                                      "register_full_backward_pre_hook"])
@pytest.mark.parametrize("part", ["ffn_norm", "moe"])
def test_hooks_on_a_submodule(part, register):
    blk = _block()
    handle = getattr(getattr(blk, part), register)(lambda *a: None)
    assert not blk._one_node()
    handle.remove()
    assert blk._one_node()


@pytest.mark.parametrize("name", ["rmsnorm", "expert_region"])
def test_replaced_operators(monkeypatch, name):
    blk = _block()
    assert blk._one_node()
    monkeypatch.setattr(F_, name, lambda *a, **kw: None)
    assert not blk._one_node()


@pytest.mark.parametrize("shape", [(6, 16), (1, 2, 3, 16), (16,)])
def test_inputs_without_three_dimensions_are_refused(shape):
    with pytest.raises(ValueError):
        _block()(torch.zeros(shape))


def test_fx_records_the_operator_of_the_norm():
    graph = torch.fx.symbolic_trace(M.RMSNorm(16)).graph
    assert torch.ops.piper_amd.rmsnorm in [n.target for n in graph.nodes]
