"""What a denoise loop forms ahead of its steps is formed only where nothing but this package's code runs between them (CPU: the kernels are stubs)."""

import pytest
import torch
import torch.nn as nn

from vllm_omni_amd import denoise, kernels
from vllm_omni_amd.blocks.flux import FluxPosEmbed, FluxTransformer2DModel
from vllm_omni_amd.cache.teacache.backend import TeaCacheBackend
from vllm_omni_amd.cache.teacache.config import TeaCacheConfig


class _OwnLinear(nn.Linear):
    pass


class _OwnPosEmbed(FluxPosEmbed):
    pass


def _hooked(m):
    m.register_forward_hook(lambda *a: None)


def _pre_hooked(m):
    m.register_forward_pre_hook(lambda *a: None)


def _wrapped(m):
    forward = m.forward
    m.forward = lambda *a, **kw: forward(*a, **kw)


_FLUX_PARTS = ["context_embedder", "time_text_embed", "time_text_embed.timestep_embedder.linear_1", "time_text_embed.guidance_embedder",
               "time_text_embed.guidance_embedder.linear_2", "time_text_embed.text_embedder", "time_text_embed.text_embedder.linear_1", "pos_embed",
               "x_embedder", "transformer_blocks.0", "transformer_blocks.0.attn.to_add_out", "single_transformer_blocks.0.proj_out", "proj_out"]


def _flux(monkeypatch):
    monkeypatch.setattr(kernels, "time_embedding", lambda embedder, t, *a: torch.zeros(t.shape[0], 64))
    monkeypatch.setattr(kernels, "project", lambda lin, x, **kw: torch.zeros(*x.shape[:-1], 64))
    return FluxTransformer2DModel(num_layers=1, num_single_layers=1, attention_head_dim=64, num_attention_heads=1, joint_attention_dim=32,
                                  pooled_projection_dim=8, axes_dims_rope=(8, 28, 28))


def _flux_steps(model):
    with torch.inference_mode():
        return model.loop_steps(torch.rand(6), torch.ones(1), torch.zeros(1, 8), torch.zeros(1, 5, 32), torch.zeros(4, 3), torch.zeros(5, 3))


def test_flux_of_its_own_classes(monkeypatch):
    model = _flux(monkeypatch)
    assert _flux_steps(model) is not None
    TeaCacheBackend(TeaCacheConfig(transformer_type="FluxTransformer2DModel", rel_l1_thresh=0.3)).enable(type("Pipe", (), {"transformer": model})())
    assert _flux_steps(model) is not None


@pytest.mark.parametrize("change", [_hooked, _pre_hooked, _wrapped])
@pytest.mark.parametrize("part", _FLUX_PARTS)
@pytest.mark.parametrize("cached", [False, True])
def test_flux_with_a_part_that_somebody_touched(monkeypatch, part, change, cached):
    model = _flux(monkeypatch)
    if cached:
        TeaCacheBackend(TeaCacheConfig(transformer_type="FluxTransformer2DModel", rel_l1_thresh=0.3)).enable(type("Pipe", (), {"transformer": model})())
    change(model.get_submodule(part))
    assert _flux_steps(model) is None


def test_flux_with_a_part_of_another_class(monkeypatch):
    for part, other in (("context_embedder", _OwnLinear(32, 64)), ("context_embedder", nn.Sequential(nn.Linear(32, 64), nn.Dropout())),
                        ("pos_embed", _OwnPosEmbed(10000, [8, 28, 28])), ("proj_out", _OwnLinear(64, 64))):
        model = _flux(monkeypatch)
        setattr(model, part, other)
        assert _flux_steps(model) is None
    model = _flux(monkeypatch)
    model.time_text_embed.text_embedder.linear_2 = nn.Sequential(nn.Linear(64, 64), nn.Dropout())
    assert _flux_steps(model) is None


class _Ahead:
    """What a loop forms ahead: a step's own number."""

    def at(self, i):
        return i


class _Recorder(nn.Module):
    """A transformer that adds the prompt's first value to the latents and notes what it is called with."""

    def __init__(self):
        super().__init__()
        self.seen, self.made = [], 0

    def loop_steps(self, timesteps, *rest):
        self.made += 1
        return _Ahead()

    def forward(self, hidden_states, encoder_hidden_states, timestep, step=None, **kw):
        self.seen.append((step, float(encoder_hidden_states.flatten()[0]), timestep.clone()))
        return (torch.zeros_like(hidden_states),)


def _flux_loop(model, prompt, n=5, on_step=None):
    denoise.diffuse_flux(model, torch.zeros(1, 4, 2), prompt, torch.zeros(1, 3), torch.zeros(4, 3), torch.zeros(2, 3), n, on_step=on_step)
    return model.seen


def test_flux_with_a_callback_between_the_steps():
    model, prompt, hooked = _Recorder(), torch.zeros(1, 2, 3), []

    def on_step(i, latents):
        prompt.fill_(i + 1)
        if i == 2:
            model.register_forward_pre_hook(lambda m, a, kw: hooked.append(sorted(kw)), with_kwargs=True)
    seen = _flux_loop(model, prompt, on_step=on_step)
    assert model.made == 0 and [s[:2] for s in seen] == [(None, float(i)) for i in range(5)]
    assert len(hooked) == 2 and all("step" not in k for k in hooked)
    other = _Recorder()
    plain = _flux_loop(other, torch.zeros(1, 2, 3))
    assert other.made == 1 and [s[0] for s in plain] == list(range(5))
    assert all(torch.equal(a[2], b[2]) for a, b in zip(seen, plain))


def test_own_tree():
    norm = FluxTransformer2DModel(num_layers=1, num_single_layers=0, attention_head_dim=64, num_attention_heads=1, joint_attention_dim=32,
                                  pooled_projection_dim=8, axes_dims_rope=(8, 28, 28))
    with torch.inference_mode():
        assert kernels.own_tree(norm) and kernels.own_tree(nn.Linear(2, 2), nn.Sequential(nn.ReLU(), nn.ModuleList()))
        layer = norm.transformer_blocks[0].attn.norm_q
        layer._forward_method = lambda x: x
        assert not kernels.own_tree(norm)
        layer._forward_method = layer.forward_hip
        assert kernels.own_tree(norm)
        around = nn.Sequential()
        around.inner = nn.Sequential(around)  # (a tree without an end)
        assert not kernels.own_tree(around)
        handle = nn.modules.module.register_module_forward_hook(lambda *a: None)
        try:
            assert not kernels.own_tree(norm)
        finally:
            handle.remove()
    assert not kernels.own_tree(norm)  # (with gradients)
