"""What is registered on the modules of a dense decoder, or on all modules, sees and
replaces what it did: the gate/up projection of an MLP is one of them, though its
product and the activation behind it may be one kernel."""
from types import SimpleNamespace

import pytest
import torch
from torch.nn.modules import module as every

from xllm_service_amd.models.llama import LlamaMLP


@pytest.fixture
def mlp():
    m = LlamaMLP(SimpleNamespace(hidden_size=16, intermediate_size=24),
                 torch.float32)
    g = torch.Generator().manual_seed(1)
    for p in m.parameters():
        p.data.normal_(generator=g)
    return m


def _register(where, m, seen):
    g = m.gate_up

    def fwd(mod, args, out):
        if mod is g:
            seen.append(1)
            return out * 0.5

    def pre(mod, args):
        if mod is g:
            seen.append(1)
            return (args[0] * 0.5,)

    def bwd(mod, *grads):
        if mod is g:
            seen.append(1)
    return {
        "forward": lambda: g.register_forward_hook(fwd),
        "forward-pre": lambda: g.register_forward_pre_hook(pre),
        "backward": lambda: g.register_full_backward_hook(bwd),
        "backward-pre": lambda: g.register_full_backward_pre_hook(bwd),
        "every forward": lambda: every.register_module_forward_hook(fwd),
        "every forward-pre": lambda: every.register_module_forward_pre_hook(pre),
        "every backward": lambda: every.register_module_full_backward_hook(bwd),
        "every backward-pre":
            lambda: every.register_module_full_backward_pre_hook(bwd),
    }[where]()


@pytest.mark.parametrize("where", [
    p + w for p in ("", "every ")
    for w in ("forward", "forward-pre", "backward", "backward-pre")])
def test_gate_up_is_seen(mlp, where):
    x = torch.randn(3, 16, generator=torch.Generator().manual_seed(2))
    x.requires_grad_(True)
    h = x @ mlp.gate_up.weight.t()
    gate, up = (h * 0.5 if "forward" in where else h).chunk(2, 1)
    want = (torch.nn.functional.silu(gate) * up) @ mlp.down.weight.t()
    seen = []
    handle = _register(where, mlp, seen)
    try:
        y = mlp(x)
        y.sum().backward()
    finally:
        handle.remove()
    assert seen
    torch.testing.assert_close(y, want, rtol=1e-4, atol=1e-4)
    seen.clear()
    mlp(x)
    assert not seen


def test_compiled_call_is_made(mlp):
    g, calls = mlp.gate_up, []
    g._compiled_call_impl = lambda *a: calls.append(1) or g._call_impl(*a)
    mlp(torch.randn(3, 16))
    assert calls
