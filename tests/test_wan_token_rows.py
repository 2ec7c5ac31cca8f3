"""Rows for the tokens of one video, by number and written out (CPU: the fused kernel is a stub)."""

import torch

from vllm_omni_amd import kernels
from vllm_omni_amd.blocks.wan import TokenRows, WanTimeTextImageEmbedding


def test_written_out_once():
    rows = TokenRows(torch.arange(12.0).view(4, 3), torch.tensor([1, 0, 0, 3, 1], dtype=torch.int32))
    assert torch.equal(rows.full(), torch.arange(12.0).view(4, 3)[[1, 0, 0, 3, 1]].unsqueeze(0))
    assert rows.full() is rows.full()  # (a block whose submodule is watched asks for it, each one)
