"""The Qwen-Image loop forms what hangs on the timestep alone for up to 16 steps at once: the latents of a loop that forms it step by step."""

import pytest
import torch

from vllm_omni_amd import denoise, kernels
from vllm_omni_amd.blocks.qwen_image import QwenImageTransformer2DModel

pytestmark = pytest.mark.gpu


class _Pipe(denoise.QwenImageCFGParallelMixin):
    def __init__(self, model):
        self.transformer, self.scheduler = model, denoise.FlowMatchEulerScheduler()


def _model(gpu, dtype, heads, D, **kw):
    g = torch.Generator(device=gpu).manual_seed(5)
    axes = (8, 28, 28) if D == 64 else (16, 56, 56)
    model = QwenImageTransformer2DModel(num_layers=2, attention_head_dim=D, num_attention_heads=heads, joint_attention_dim=256, axes_dims_rope=axes, **kw).to(device=gpu, dtype=dtype)
    with torch.no_grad():
        for p in model.parameters():
            p.normal_(0.0, 0.05, generator=g)
    model.fuse_modulation()
    return model


def _args(gpu, dtype, steps, neg, seed=1):
    g = torch.Generator(device=gpu).manual_seed(seed)
    rand = lambda *s: torch.randn(*s, device=gpu, generator=g).to(dtype)  # noqa: E731
    return dict(prompt_embeds=rand(1, 30, 256), prompt_embeds_mask=None, negative_prompt_embeds=rand(1, neg, 256) if neg else None, negative_prompt_embeds_mask=None,
                latents=rand(1, 96, 64), img_shapes=[[(1, 12, 8)]], txt_seq_lens=[30], negative_txt_seq_lens=[neg] if neg else None, timesteps=steps, do_true_cfg=neg > 0,
                guidance=None, true_cfg_scale=2.0)


# (up to 4 steps of a multiple of 512 channels: the stream kernel, as for one step; more: the matrix kernel, another order of summation)
@pytest.mark.parametrize("heads,D,n,neg,same", [(4, 64, 1, 0, True), (4, 64, 4, 9, True), (3, 128, 17, 30, True), (4, 128, 4, 9, True), (4, 128, 1, 30, True), (4, 128, 18, 9, False)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_loop(gpu, monkeypatch, heads, D, n, neg, same, dtype):
    print(f"loop of {n} steps, {heads} x {D}, negative {neg} {dtype}", flush=True)
    pipe = _Pipe(_model(gpu, dtype, heads, D))
    pipe.scheduler.set_timesteps(max(n, 20), device=gpu, mu=0.8)
    args = _args(gpu, dtype, pipe.scheduler.timesteps[:n], neg)
    seen = []
    real = QwenImageTransformer2DModel.steps_rows
    monkeypatch.setattr(QwenImageTransformer2DModel, "steps_rows", lambda self, t: seen.append(t.shape[0]) or real(self, t))
    with torch.inference_mode():
        got = pipe.diffuse(**args)
        assert seen == [min(16, n - i) for i in range(0, n, 16)]
        monkeypatch.setattr(QwenImageTransformer2DModel, "steps_rows", lambda self, t: None)
        want = pipe.diffuse(**args)
    assert bool(torch.isfinite(want.float()).all())
    if same:
        assert torch.equal(got, want)
    else:  # conditioning rows whose float32 sums round the other way here and there: far below a rounding of every latent in every step
        assert float((got.float() - want.float()).norm()) < n * (2.0 ** -9 if dtype == torch.bfloat16 else 2.0 ** -12) * float(want.float().norm())


def test_not_taken(gpu, monkeypatch):
    """Whoever stands between the loop and the model gets the calls as ever."""
    pipe = _Pipe(_model(gpu, torch.bfloat16, 4, 64))
    pipe.scheduler.set_timesteps(20, device=gpu, mu=0.8)
    args = _args(gpu, torch.bfloat16, pipe.scheduler.timesteps[:2], 0)
    with torch.inference_mode():
        want = pipe.diffuse(**args)
        seen = []
        forward = type(pipe.transformer).forward
        pipe.transformer.forward = lambda **kw: seen.append(sorted(kw)) or forward(pipe.transformer, **kw)
        assert torch.equal(pipe.diffuse(**args), want) and len(seen) == 2 and all("step" not in k for k in seen)
        del pipe.transformer.forward
        pipe.predict_noise = lambda **kw: seen.append(sorted(kw)) or pipe.transformer(**kw)[0]
        assert torch.equal(pipe.diffuse(**args), want) and len(seen) == 4 and all("step" not in k for k in seen)
        del pipe.predict_noise
        handle = pipe.transformer.time_text_embed.register_forward_hook(lambda m, a, out: seen.append("hook"))
        assert torch.equal(pipe.diffuse(**args), want) and seen[4:] == ["hook"] * 2
        handle.remove()
        pipe.transformer._mod_weight = None
        assert pipe.transformer.steps_rows(torch.rand(2, device=gpu).bfloat16()) is None
        edit = _model(gpu, torch.bfloat16, 4, 64, zero_cond_t=True)
        assert edit.steps_rows(torch.rand(2, device=gpu).bfloat16()) is None and pipe.transformer.steps_rows(torch.rand(2, device=gpu)) is None
        assert kernels.native_blocks()
    plain = _model(gpu, torch.bfloat16, 4, 64)
    assert plain.steps_rows(torch.rand(2, device=gpu).bfloat16()) is None  # with gradients
