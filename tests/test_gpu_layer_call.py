"""A layer's call (layers/custom_op.py): at once the native one only where a module's call would come to nothing else, and then the same result; hooks, replaced methods
and classes, compiled modules, traces and a replaced way of calling modules are seen by torch as ever."""

import pickle
import sys

import pytest
import torch
import torch.nn as nn

from vllm_omni_amd import kernels
from vllm_omni_amd.layers.adalayernorm import AdaLayerNorm
from vllm_omni_amd.layers.rmsnorm import RMSNorm
from vllm_omni_amd.layers.rope import RotaryEmbedding

pytestmark = pytest.mark.gpu


def _layers(gpu):
    g = torch.Generator(device=gpu).manual_seed(1)
    r = lambda *s: torch.randn(*s, device=gpu, generator=g).bfloat16()
    return [(RMSNorm(128).to(device=gpu, dtype=torch.bfloat16), (r(1, 5, 4, 128),)), (AdaLayerNorm(256).to(gpu), (r(1, 5, 256), r(1, 768))),
            (RotaryEmbedding(), (r(1, 5, 4, 64), torch.rand(5, 32, device=gpu, generator=g), torch.rand(5, 32, device=gpu, generator=g)))]


def _at_once(layer, args):
    """Whether a call goes down without torch's."""
    return kernels.native().layer_call(layer, *args) is not None


def _equal(a, b):
    return all(torch.equal(x, y) for x, y in zip(*(t if isinstance(t, tuple) else (t,) for t in (a, b))))


@pytest.mark.parametrize("which", [0, 1, 2])
def test_call(gpu, which, monkeypatch):
    layer, args = _layers(gpu)[which]
    cls = type(layer)
    with torch.inference_mode():
        want = layer.forward(*args)
        assert _at_once(layer, args) and _equal(layer(*args), want)
        again = pickle.loads(pickle.dumps(layer))
        assert _at_once(again, args) and _equal(again(*args), want)

        seen = []
        note = lambda *a: seen.append(1)
        for register in (layer.register_forward_hook, layer.register_forward_pre_hook, layer.register_full_backward_hook, layer.register_full_backward_pre_hook,
                         nn.modules.module.register_module_forward_hook, nn.modules.module.register_module_forward_pre_hook,
                         nn.modules.module.register_module_full_backward_hook, nn.modules.module.register_module_full_backward_pre_hook):
            hook = register(note)
            assert not _at_once(layer, args) and _equal(layer(*args), want)
            hook.remove()
            assert _at_once(layer, args)
        assert len(seen) == 4  # (the forward ones)

        own = lambda *a, **k: "own"
        for name in ("forward", "_call_impl"):
            layer.__dict__[name] = own
            assert layer(*args) == "own"
            del layer.__dict__[name]
        layer._forward_method = own
        assert layer(*args) == "own"
        del layer.__dict__["_forward_method"]
        layer._forward_method = layer.forward_hip
        layer._compiled_call_impl = own
        assert layer(*args) == "own"
        layer._compiled_call_impl = None
        assert _at_once(layer, args)
        for where, name in ((cls, "forward"), (nn.Module, "__call__"), (nn.Module, "_call_impl")):
            with monkeypatch.context() as m:
                m.setattr(where, name, own)
                assert layer(*args) == "own"
        sub = type("Sub", (cls,), {"forward": own}).__new__(type("Sub", (cls,), {"forward": own}))
        sub.__dict__.update(layer.__dict__)
        assert sub(*args) == "own"
        assert _equal(layer(*args), want)
    assert not _at_once(layer, (args[0].cpu(), *args[1:]))


def test_traces(gpu):
    layer, args = _layers(gpu)[0]
    during = []

    class Model(nn.Module):
        def __init__(self):
            super().__init__()
            self.norm = layer

        def forward(self, x):
            if torch.jit.is_tracing():
                during.append(_at_once(self.norm, (x,)))
            return self.norm(x) * 2

    with torch.inference_mode():
        want = Model()(*args)
        torch.jit.trace(Model(), args, check_trace=False)
        assert during == [False]

        class Tracer(torch.fx.Tracer):
            def is_leaf_module(self, m, name):
                return m is layer or super().is_leaf_module(m, name)

        graph = Tracer().trace(_Plain(layer))
        assert [n.target for n in graph.nodes if n.op == "call_module"] == ["norm"]
        assert torch.equal(want, layer(*args) * 2)


class _Plain(nn.Module):
    def __init__(self, norm):
        super().__init__()
        self.norm = norm

    def forward(self, x):
        return self.norm(x) * 2


@pytest.mark.parametrize("which", [0, 1, 2])
def test_replaced_on_any_class(gpu, which, monkeypatch):
    """torch looks for its ways of calling a module in all of the layer's classes."""
    from vllm_omni_amd.layers.custom_op import CustomOp

    layer, args = _layers(gpu)[which]
    own = lambda *a, **k: "own"
    with torch.inference_mode():
        want = layer.forward(*args)
        for cls in (type(layer), CustomOp, nn.Module):
            for name in ("_call_impl", "_compiled_call_impl"):
                with monkeypatch.context() as m:
                    m.setattr(cls, name, own, raising=False)
                    assert not _at_once(layer, args)
                    assert layer(*args) == "own"
                assert _at_once(layer, args) and _equal(layer(*args), want)


@pytest.mark.parametrize("which", [0, 1, 2])
def test_calls_that_are_followed(gpu, which, tmp_path):
    """A profiler or debugger of the thread sees torch's call of the module and the layer's forward."""
    layer, args = _layers(gpu)[which]
    for follow in (sys.setprofile, sys.settrace):
        calls = []
        before = sys.gettrace() if follow is sys.settrace else sys.getprofile()
        with torch.inference_mode():
            follow(lambda frame, event, arg: calls.append(frame.f_code.co_name) if event == "call" else None)
            layer(*args)
            follow(before)
        assert "_call_impl" in calls and "forward" in calls, calls
    with torch.inference_mode(), torch.profiler.profile(activities=[torch.profiler.ProfilerActivity.CPU], with_stack=True) as p:
        layer(*args)
    p.export_chrome_trace(str(tmp_path / "trace.json"))
    assert f"nn.Module: {type(layer).__name__}" in (tmp_path / "trace.json").read_text()
    with torch.inference_mode():
        assert _at_once(layer, args)
