"""A layer's own call takes what it holds from the layer as it is at the call, and only where class and method are this package's."""

import copy

import pytest
import torch

from vllm_omni_amd.layers.adalayernorm import AdaLayerNorm
from vllm_omni_amd.layers.rmsnorm import RMSNorm
from vllm_omni_amd.layers.rope import RotaryEmbedding

pytestmark = pytest.mark.gpu


def _cases(gpu, dtype):
    g = torch.Generator(device=gpu).manual_seed(2)
    rand = lambda *s: torch.randn(*s, device=gpu, generator=g)  # noqa: E731
    x, h = rand(2, 33, 512).to(dtype), rand(2, 33, 4, 128).to(dtype)
    a = rand(33, 64)
    norm = RMSNorm(128).to(device=gpu, dtype=dtype)
    with torch.no_grad():
        norm.weight.copy_(rand(128))
    return [(norm, (h,)), (RotaryEmbedding(), (h, a.cos(), a.sin())), (RotaryEmbedding(is_neox_style=True), (h, a.cos(), a.sin())),
            (RotaryEmbedding(), (h, a.cos()[None], a.sin()[None])), (AdaLayerNorm(512), (x, rand(2, 1536).to(dtype))),
            (AdaLayerNorm(512, elementwise_affine=True).to(gpu), (x, rand(2, 1536).to(dtype))), (AdaLayerNorm(512, ref_rounding=True), (x, rand(2, 1536).to(dtype))),
            (AdaLayerNorm(512), (x, rand(4, 1536).to(dtype), torch.randint(2, (2, 33), device=gpu, dtype=torch.int32)))]


def _same(a, b):
    return all(torch.equal(p, q) for p, q in zip(a, b, strict=True)) if isinstance(a, tuple) else torch.equal(a, b)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("at", range(8))
def test_calls(gpu, dtype, at):
    with torch.inference_mode():
        layer, args = _cases(gpu, dtype)[at]
        want = layer.forward_hip(*args)
        assert _same(layer(*args), want) and _same(copy.deepcopy(layer)(*args), want)
        names = ("x", "cos", "sin") if isinstance(layer, RotaryEmbedding) else ("x", "mod_params", "index")
        assert _same(layer(**dict(zip(names, args))), want)


def test_results_are_as_torch_makes_them(gpu):
    layer, args = _cases(gpu, torch.bfloat16)[1]
    for mode in (torch.inference_mode, torch.no_grad):
        with mode():
            out, like = layer(*args), torch.empty_like(args[0])
        assert out.is_inference() == like.is_inference() and not out.requires_grad and out.device == like.device and out.stride() == like.stride()


def test_layer_as_it_is(gpu):
    with torch.inference_mode():
        norm, (h,) = _cases(gpu, torch.bfloat16)[0]
        before = norm(h)
        norm.weight.data = norm.weight.data * 2
        assert torch.equal(norm(h), norm.forward_hip(h)) and not torch.equal(norm(h), before)
        norm.variance_epsilon = 1.0
        assert torch.equal(norm(h), norm.forward_hip(h))
        rope, args = _cases(gpu, torch.bfloat16)[1]
        rope.is_neox_style = True
        assert torch.equal(rope(*args), rope.forward_hip(*args))
        ada, args = _cases(gpu, torch.bfloat16)[4]
        ada.eps = 0.5
        assert _same(ada(*args), ada.forward_hip(*args))
        with pytest.raises(ValueError):
            ada(args[0][..., :256], args[1])
        with pytest.raises(ValueError):
            norm(h[..., :64])
        # another method, another class, a hook
        for layer, a in _cases(gpu, torch.bfloat16):
            layer._forward_method = lambda *x: "mine"
            assert layer(*a) == "mine"

        class Mine(RMSNorm):
            def forward_hip(self, x):
                return "mine"
        assert Mine(128).to(device=gpu, dtype=torch.bfloat16)(h) == "mine"
        norm.register_forward_hook(lambda m, a, out: "seen")
        assert norm(h) == "seen"
