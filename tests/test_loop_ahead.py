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


class _Qwen(nn.Module):
    def __init__(self, number):
        super().__init__()
        self.number, self.seen = number, []

    def steps_rows(self, timesteps):
        return [(self.number, float(t)) for t in timesteps]

    def forward(self, hidden_states, timestep, step=None, **kw):
        self.seen.append((step, timestep.clone()))
        return (torch.zeros_like(hidden_states),)


class _Pipe(denoise.QwenImageCFGParallelMixin):
    def __init__(self, scheduler=None):
        self.transformer, self.scheduler = _Qwen(0), scheduler or denoise.FlowMatchEulerScheduler()


def _qwen_loop(pipe, n=5):
    pipe.scheduler.set_timesteps(n)
    steps = pipe.scheduler.timesteps
    pipe.diffuse(torch.zeros(1, 3, 2), None, None, None, torch.zeros(1, 4, 2), [], [3], None, steps, False, None, 1.0)
    return [float(t) for t in steps]


def test_qwen_ahead(monkeypatch):
    monkeypatch.setattr(kernels, "own_tree", lambda m: True)
    pipe = _Pipe()
    steps = _qwen_loop(pipe, 18)
    # (up to 16 at once)
    assert [s for s, _ in pipe.transformer.seen] == [(0, pytest.approx(t / 1000)) for t in steps]
    assert all(torch.equal(t, torch.tensor([s]) / 1000) for (_, t), s in zip(pipe.transformer.seen, steps))


class _OwnScheduler(denoise.FlowMatchEulerScheduler):
    def step(self, *a, **kw):
        self.between()
        return super().step(*a, **kw)


class _OwnStep(_Pipe):
    def scheduler_step(self, *a):
        self.between()
        return super().scheduler_step(*a)


class _OwnCombination(_Pipe):
    def combine_cfg_noise(self, *a):
        return super().combine_cfg_noise(*a)


class _OwnSwitch(_Pipe):
    interrupt = property(lambda self: self.between())


@pytest.mark.parametrize("how", ["scheduler", "scheduler's method", "step", "own step", "switch"])
def test_qwen_with_somebody_elses_code_between_the_steps(monkeypatch, how):
    """It exchanges the transformer, writes to the timesteps and registers a hook on the second one."""
    monkeypatch.setattr(kernels, "own_tree", lambda m: True)
    kind = {"own step": _OwnStep, "switch": _OwnSwitch}.get(how, _Pipe)
    pipe = kind(_OwnScheduler() if how == "scheduler" else None)
    first, second, hooked, calls = pipe.transformer, _Qwen(1), [], []

    def between():
        calls.append(1)
        if len(calls) == 3:
            pipe.transformer = second
            pipe.scheduler.timesteps[-1] = 7.0
            second.register_forward_pre_hook(lambda m, a, kw: hooked.append(sorted(kw)), with_kwargs=True)
    if how == "scheduler's method":
        real = pipe.scheduler.step
        pipe.scheduler.step = lambda *a, **kw: between() or real(*a, **kw)
    elif how == "step":
        real = pipe.scheduler_step
        pipe.scheduler_step = lambda *a: between() or real(*a)
    pipe.between = pipe.scheduler.between = between
    _qwen_loop(pipe)
    seen = first.seen + second.seen
    assert len(seen) == 5 and len(second.seen) >= 2 and all(s is None for s, _ in seen)
    assert torch.equal(seen[-1][1], torch.tensor([7.0]) / 1000) and len(hooked) == len(second.seen) and all("step" not in k for k in hooked)


def test_qwen_own_steps():
    assert _Pipe()._own_steps() and not _OwnCombination()._own_steps() and not _OwnSwitch()._own_steps()
    pipe = _Pipe()
    pipe.interrupt = True
    assert pipe._own_steps()
    with torch.inference_mode():
        assert not kernels.own_tree(pipe.transformer)  # (a class of this file)


def test_flux_forms_each_timestep_once(monkeypatch):
    """Also where the model forms nothing ahead."""
    model, made, full = _Recorder(), [], torch.full
    model.loop_steps = lambda *a: None
    monkeypatch.setattr(denoise.torch, "full", lambda *a, **kw: made.append(a) or full(*a, **kw))
    _flux_loop(model, torch.zeros(1, 2, 3))
    assert sum(1 for a in made if a[1] != 3.5) == 5


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
