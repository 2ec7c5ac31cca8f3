"""Rows for the tokens of one video, by number and written out (CPU: the fused kernel is a stub)."""

import torch

from vllm_omni_amd import kernels
from vllm_omni_amd.blocks.wan import TokenRows, WanTimeTextImageEmbedding


def test_written_out_once():
    rows = TokenRows(torch.arange(12.0).view(4, 3), torch.tensor([1, 0, 0, 3, 1], dtype=torch.int32))
    assert torch.equal(rows.full(), torch.arange(12.0).view(4, 3)[[1, 0, 0, 3, 1]].unsqueeze(0))
    assert rows.full() is rows.full()  # (a block whose submodule is watched asks for it, each one)


def test_a_caller_without_rows_by_number(monkeypatch):
    """Who takes the rows of all tokens gets them as they are formed, not formed by number and written out."""
    asked = []
    monkeypatch.setattr(kernels, "time_tokens", lambda *a: asked.append(a) or (torch.zeros(4, 8), torch.zeros(4, 48), torch.zeros(4, dtype=torch.int32)))
    monkeypatch.setattr(kernels, "project", lambda lin, x, **kw: torch.zeros(*x.shape[:-1], lin.out_features))
    monkeypatch.setattr(kernels, "gelu_tanh", lambda x, out=None: x)
    embed = WanTimeTextImageEmbedding(dim=8, time_freq_dim=16, time_proj_dim=48, text_embed_dim=4)
    args = (torch.rand(4), torch.zeros(1, 3, 4))
    with torch.inference_mode():
        temb, proj, *_ = embed(*args, timestep_seq_len=4)
        assert not asked and temb.shape == (1, 4, 8) and proj.shape == (1, 4, 48)
        temb, proj, *_ = embed(*args, timestep_seq_len=4, token_rows=True)
        assert len(asked) == 1 and isinstance(temb, TokenRows) and isinstance(proj, TokenRows)
