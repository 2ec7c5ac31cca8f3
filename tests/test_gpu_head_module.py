"""The head's norm and projection as modules (AdaLayerNormContinuous.head): one launch only where both are plainly what their classes say; what a program has put on a
module, on the class or in a module's place takes effect."""

import pytest
import torch
import torch.nn as nn

from vllm_omni_amd import kernels
from vllm_omni_amd.blocks.qwen_image import AdaLayerNormContinuous

pytestmark = pytest.mark.gpu


def _modules(gpu):
    torch.manual_seed(3)
    norm = AdaLayerNormContinuous(3072, 3072).to(device=gpu, dtype=torch.bfloat16)
    lin = nn.Linear(3072, 64, device=gpu, dtype=torch.bfloat16)
    x, cond = torch.randn(2, 70, 3072, device=gpu).bfloat16(), torch.randn(2, 3072, device=gpu).bfloat16()
    return norm, lin, x, cond


def _close(a, b):
    return float((a.double() - b.double()).norm() / b.double().norm()) < 2.0 ** -8  # (sums in another order, rounded twice)


@pytest.mark.parametrize("given", [False, True])
def test_head(gpu, monkeypatch, given):
    """``given``: with the projection of the condition at hand, which a module's own forward has no part in."""
    norm, lin, x, cond = _modules(gpu)
    launches = []
    normed = kernels.project_normed
    monkeypatch.setattr(kernels, "project_normed", lambda *a: launches.append(normed(*a)) or launches[-1])
    with torch.inference_mode():
        emb = kernels.project(norm.linear, cond, silu_input=True)
        head = lambda: AdaLayerNormContinuous.head(norm, lin, x, cond, emb if given else None)  # noqa: E731
        want = lin(norm(x, cond))

        def at_once():
            launches.clear()
            out = head()
            return out, bool(launches) and launches[-1] is not None

        out, one = at_once()
        assert one and _close(out, want)

        def replaced(result):
            out, one = at_once()
            assert not one and torch.equal(out, result)

        # on the class, on the module
        twice = lambda self, x, emb: 2 * x  # noqa: E731
        for put in (lambda m: m.setattr(AdaLayerNormContinuous, "modulate", twice), lambda m: m.setitem(norm.__dict__, "modulate", lambda x, emb: 2 * x)):
            with monkeypatch.context() as m:
                put(m)
                replaced(lin(2 * x))
        if not given:
            for put in (lambda m: m.setattr(AdaLayerNormContinuous, "forward", lambda self, x, cond: 3 * x), lambda m: m.setitem(norm.__dict__, "forward", lambda x, cond: 3 * x)):
                with monkeypatch.context() as m:
                    put(m)
                    replaced(lin(3 * x))
            hook = norm.register_forward_hook(lambda mod, a, o: 4 * x)
            replaced(lin(4 * x))
            hook.remove()
            hook = norm.linear.register_forward_hook(lambda mod, a, o: o * 0)  # (no scale, no shift: one launch of the hook's rows is as good)
            out = head()
            assert _close(out, lin(torch.nn.functional.layer_norm(x.float(), (3072,), eps=norm.eps).bfloat16()))
            hook.remove()
            assert _close(AdaLayerNormContinuous.head(norm, lin, x, cond.float()), lin(norm(x, cond.float())))  # another type of condition

            class Other(nn.Module):
                def forward(self, x, cond):
                    return 5 * x

            assert torch.equal(AdaLayerNormContinuous.head(Other(), lin, x, cond), lin(5 * x))

        # the projection: hooked, and in a wrapper of somebody else's
        hook = lin.register_forward_hook(lambda mod, a, o: o + 1)
        out, one = at_once()
        assert not one and _close(out - 1, want)
        hook.remove()

        class Wrapped(nn.Linear):
            def forward(self, x):
                return super().forward(x) * 2

        lin = Wrapped(3072, 64, device=gpu, dtype=torch.bfloat16)
        out, one = at_once()
        assert not one and torch.equal(out, lin(norm(x, cond)))
