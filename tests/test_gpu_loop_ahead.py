"""Both loops with somebody else's code between or inside their steps: the latents of a loop that forms everything in every step."""

import pytest
import torch

from vllm_omni_amd import denoise
from vllm_omni_amd.blocks.flux import FluxTransformer2DModel
from vllm_omni_amd.blocks.qwen_image import QwenImageTransformer2DModel

pytestmark = pytest.mark.gpu


def _filled(model, gpu, seed):
    g = torch.Generator(device=gpu).manual_seed(seed)
    model = model.to(device=gpu, dtype=torch.bfloat16)
    with torch.no_grad():
        for p in model.parameters():
            p.normal_(0.0, 0.05, generator=g)
    model.fuse_modulation()
    return model


def _rand(gpu, *shape):
    return torch.randn(*shape, device=gpu, generator=torch.Generator(device=gpu).manual_seed(sum(shape))).to(torch.bfloat16)


def _flux(gpu):
    return _filled(FluxTransformer2DModel(num_layers=1, num_single_layers=1, attention_head_dim=64, num_attention_heads=4, joint_attention_dim=256,
                                          pooled_projection_dim=128, axes_dims_rope=(8, 28, 28)), gpu, 5)


def _qwen(gpu, seed):
    return _filled(QwenImageTransformer2DModel(num_layers=2, attention_head_dim=64, num_attention_heads=4, joint_attention_dim=256,
                                               axes_dims_rope=(8, 28, 28)), gpu, seed)


def _flux_loop(gpu, change, forced):
    model, prompt = _flux(gpu), _rand(gpu, 1, 30, 256)
    if forced:
        model.loop_steps = lambda *a: None
    ids = torch.zeros(96, 3, device=gpu)
    ids[:, 1] = torch.arange(96, device=gpu)
    return denoise.diffuse_flux(model, _rand(gpu, 1, 96, 64), prompt, _rand(gpu, 1, 128), ids, torch.zeros(30, 3, device=gpu), 4, on_step=change(model, prompt))


def _prompt_written(model, prompt):
    return lambda i, latents: prompt.mul_(1.5)


def _weight_written(model, prompt):
    return lambda i, latents: model.time_text_embed.timestep_embedder.linear_2.weight.data.mul_(2.0)


def _adapter_by_step(model, prompt):
    calls = []
    model.context_embedder.register_forward_hook(lambda m, a, out: out * (1.0 + 0.5 * (calls.append(1) or len(calls))))
    return None


@pytest.mark.parametrize("change", [_prompt_written, _weight_written, _adapter_by_step])
def test_flux(gpu, change):
    print(f"flux loop, {change.__name__}", flush=True)
    with torch.inference_mode():
        got, want, still = _flux_loop(gpu, change, False), _flux_loop(gpu, change, True), _flux_loop(gpu, lambda *a: None, False)
    assert bool(torch.isfinite(got.float()).all()) and torch.equal(got, want) and not torch.equal(got, still)


class _Pipe(denoise.QwenImageCFGParallelMixin):
    def __init__(self, model):
        self.transformer, self.scheduler = model, denoise.FlowMatchEulerScheduler()


class _TwoExperts(_Pipe):
    def scheduler_step(self, noise, t, latents):
        if self.other is not None:
            self.transformer, self.other = self.other, None
        return super().scheduler_step(noise, t, latents)


def test_qwen_with_two_transformers(gpu):
    print("qwen loop, two transformers", flush=True)
    got = []
    with torch.inference_mode():
        for forced in (False, True):
            pipe = _TwoExperts(_qwen(gpu, 5))
            pipe.other = _qwen(gpu, 6)
            if forced:
                pipe.transformer.steps_rows = pipe.other.steps_rows = lambda t: None
            pipe.scheduler.set_timesteps(4, device=gpu, mu=0.8)
            got.append(pipe.diffuse(_rand(gpu, 1, 30, 256), None, _rand(gpu, 1, 9, 256), None, _rand(gpu, 1, 96, 64), [[(1, 12, 8)]], [30], [9],
                                    pipe.scheduler.timesteps, True, None, 2.0))
        pipe = _Pipe(_qwen(gpu, 5))
        pipe.scheduler.set_timesteps(4, device=gpu, mu=0.8)
        one = pipe.diffuse(_rand(gpu, 1, 30, 256), None, _rand(gpu, 1, 9, 256), None, _rand(gpu, 1, 96, 64), [[(1, 12, 8)]], [30], [9],
                           pipe.scheduler.timesteps, True, None, 2.0)
    assert bool(torch.isfinite(got[0].float()).all()) and torch.equal(got[0], got[1]) and not torch.equal(got[0], one)
