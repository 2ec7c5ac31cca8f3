"""A layer's call that is not of the native form costs no memory on its way to the form that takes it."""

import pytest
import torch

from vllm_omni_amd.layers.rope import RotaryEmbedding

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("form,made", [("dense", 1), ("strided", 2), ("tables", 3)])  # the result; with a dense copy; with the tables in float32
def test_rotary_allocations(gpu, form, made):
    layer, a = RotaryEmbedding(), torch.rand(33, 64, device=gpu)
    x = torch.randn(2, 33, 4, 256 if form == "strided" else 128, device=gpu, dtype=torch.bfloat16)[..., :128]
    dtype = torch.bfloat16 if form == "tables" else torch.float32
    cos, sin = a.cos().to(dtype), a.sin().to(dtype)
    with torch.inference_mode():
        layer(x, cos, sin)
        before = torch.cuda.memory_stats()["allocation.all.allocated"]
        out = layer(x, cos, sin)
        assert torch.cuda.memory_stats()["allocation.all.allocated"] - before == made
        want = RotaryEmbedding()(x.contiguous(), cos.float(), sin.float())
    assert torch.equal(out, want)
