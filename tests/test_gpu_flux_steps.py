"""The Flux loop forms text tokens, rotary tables and conditioning once: the latents and the decisions of a loop that forms them in every step."""

import pytest
import torch

from vllm_omni_amd import denoise
from vllm_omni_amd.blocks.flux import FluxTransformer2DModel
from vllm_omni_amd.cache.teacache.backend import TeaCacheBackend
from vllm_omni_amd.hooks.base import HookRegistry, ModelHook

pytestmark = pytest.mark.gpu


def _model(gpu, dtype, heads=4, D=64, dual=2, single=2):
    g = torch.Generator(device=gpu).manual_seed(5)
    model = FluxTransformer2DModel(num_layers=dual, num_single_layers=single, attention_head_dim=D, num_attention_heads=heads, joint_attention_dim=256,
                                   pooled_projection_dim=128, axes_dims_rope=(8, 28, 28) if D == 64 else (16, 56, 56)).to(device=gpu, dtype=dtype)
    with torch.no_grad():
        for p in model.parameters():
            p.normal_(0.0, 0.05, generator=g)
    model.fuse_modulation()
    return model


def _args(gpu, dtype, n):
    g = torch.Generator(device=gpu).manual_seed(1)
    rand = lambda *s: torch.randn(*s, device=gpu, generator=g).to(dtype)  # noqa: E731
    ids = torch.zeros(96, 3, device=gpu)
    ids[:, 1], ids[:, 2] = torch.arange(96, device=gpu) // 8, torch.arange(96, device=gpu) % 8
    return dict(latents=rand(1, 96, 64), prompt_embeds=rand(1, 30, 256), pooled_prompt_embeds=rand(1, 128), img_ids=ids, txt_ids=torch.zeros(30, 3, device=gpu),
                num_inference_steps=n)


@pytest.mark.parametrize("heads,D,dual,single,n", [(4, 64, 2, 2, 1), (4, 64, 2, 2, 2), (4, 64, 0, 3, 9), (4, 128, 2, 0, 5), (4, 128, 1, 1, 8)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("cached", [False, True])
def test_loop(gpu, monkeypatch, heads, D, dual, single, n, dtype, cached):
    if cached and dual == 0:
        pytest.skip("the cache looks at the first dual block")
    print(f"flux loop {heads}x{D} {dual}+{single} n={n} {dtype} cached={cached}", flush=True)
    model, args, got, decisions = _model(gpu, dtype, heads, D, dual, single), _args(gpu, dtype, n), [], []
    pipe = type("Pipe", (), {"transformer": model})()
    backend = None
    if cached:
        from vllm_omni_amd.cache.teacache.config import TeaCacheConfig

        backend = TeaCacheBackend(TeaCacheConfig(transformer_type="FluxTransformer2DModel", rel_l1_thresh=0.3))
        backend.enable(pipe)
    made = []
    real = FluxTransformer2DModel.loop_steps
    with torch.inference_mode():
        for f in (lambda self, *a: made.append(real(self, *a)) or made[-1], lambda self, *a: None):
            monkeypatch.setattr(FluxTransformer2DModel, "loop_steps", f)
            if cached:
                backend.refresh(pipe, n)
            got.append(denoise.diffuse_flux(model, **args))
            if cached:
                decisions.append([d["compute"] for d in model._hook_registry.get_hook("teacache").decisions[-n:]])
    assert len(made) == (n > 1) and all(s is not None and s.fused == (not cached) for s in made)
    assert bool(torch.isfinite(got[0].float()).all()) and torch.equal(got[0], got[1]) and (not cached or decisions[0] == decisions[1])


def test_not_taken(gpu):
    model, args = _model(gpu, torch.bfloat16), _args(gpu, torch.bfloat16, 2)
    with torch.inference_mode():
        want = denoise.diffuse_flux(model, **args)
        seen = []
        handle = model.register_forward_pre_hook(lambda m, a, kw: seen.append(sorted(kw)), with_kwargs=True)
        assert torch.equal(denoise.diffuse_flux(model, **args), want) and len(seen) == 2 and all("step" not in k for k in seen)
        handle.remove()

        class Watch(ModelHook):
            def new_forward(self, module, *a, **kw):
                seen.append(sorted(kw))
                return module._original_forward(*a, **kw)
        HookRegistry.get_or_create(model).register_hook("watch", Watch())
        assert torch.equal(denoise.diffuse_flux(model, **args), want) and len(seen) == 4 and all("step" not in k for k in seen)
        other = _model(gpu, torch.bfloat16)
        other.time_text_embed.register_forward_hook(lambda *a: seen.append("hook"))
        assert torch.equal(denoise.diffuse_flux(other, **args), want) and seen[4:] == ["hook"] * 2
