"""A timestep projection of somebody else's is the one that the embedding is made from (CPU: the fused kernel is a stub)."""

import pytest
import torch

from vllm_omni_amd import kernels
from vllm_omni_amd.blocks.qwen_image import QwenImageTransformer2DModel, QwenTimestepProjEmbeddings


class _Mine(QwenTimestepProjEmbeddings):
    @staticmethod
    def time_proj(t, dim=256, max_period=10000, scale=1000.0, dtype=torch.float32, pre=1.0):
        return torch.full((t.shape[0], dim), 2.0, dtype=dtype)


@pytest.mark.parametrize("how", ["class", "instance", "none"])
def test_time_proj(monkeypatch, how):
    monkeypatch.setattr(kernels, "time_embedding", lambda embedder, t, *a: torch.zeros(t.shape[0], 64))
    embed = (_Mine if how == "class" else QwenTimestepProjEmbeddings)(64)
    if how == "instance":
        embed.time_proj = _Mine.time_proj
    fed = []
    embed.timestep_embedder.forward = lambda x, **kw: fed.append(x) or x[:, :64]
    with torch.inference_mode():
        out = embed(torch.tensor([0.3, 0.7]), torch.zeros(2, 5, 64))
        model = QwenImageTransformer2DModel(num_layers=1, attention_head_dim=64, num_attention_heads=1, joint_attention_dim=64, axes_dims_rope=(8, 28, 28))
        model.fuse_modulation()
        model.time_text_embed = embed
        monkeypatch.setattr(kernels, "linear_few_pair", lambda x, w, b, lin: (torch.zeros(x.shape[0], w.shape[0]), torch.zeros(x.shape[0], 128)))
        rows = model.steps_rows(torch.tensor([0.3, 0.7]))
    if how == "none":
        assert not fed and torch.equal(out, torch.zeros(2, 64)) and len(rows) == 2
    else:
        assert len(fed) == 1 and torch.equal(fed[0], torch.full((2, 256), 2.0)) and torch.equal(out, torch.full((2, 64), 2.0)) and rows is None
