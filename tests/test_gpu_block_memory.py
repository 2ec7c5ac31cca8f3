"""A native block's intermediate tensors share memory where the per-kernel path frees one before it makes the next."""

import gc

import pytest
import torch

from test_gpu_native_path import _init
from vllm_omni_amd import kernels

pytestmark = pytest.mark.gpu


def _wan(gpu, per_token):
    from vllm_omni_amd.blocks.wan import WanTransformer3DModel

    model = _init(WanTransformer3DModel(num_attention_heads=4, attention_head_dim=64, text_dim=128, ffn_dim=704, num_layers=2), gpu,
                  torch.bfloat16)
    video, text = torch.randn(2, 16, 8, 60, 66, device=gpu).bfloat16(), torch.randn(2, 40, 128, device=gpu).bfloat16()
    t = torch.full((2, 8 * 30 * 33) if per_token else (2,), 500.0, device=gpu)
    x, ctx, temb, tproj, rotary = model.prepare(video, t, text)
    return 2 * 8 * 30 * 33 * 256 * 2, lambda: model.run_blocks(x, ctx, tproj, rotary)


def _qwen(gpu, txt):
    from vllm_omni_amd.blocks.qwen_image import QwenImageTransformer2DModel

    model = _init(QwenImageTransformer2DModel(num_layers=2, attention_head_dim=64, num_attention_heads=4, joint_attention_dim=256,
                                              axes_dims_rope=(8, 28, 28)), gpu, torch.bfloat16)
    model.fuse_modulation()
    lat, enc = torch.randn(2, 64 * 64, 64, device=gpu).bfloat16(), torch.randn(2, txt, 256, device=gpu).bfloat16()
    t = torch.full((2,), 0.3, device=gpu).bfloat16()
    img, text, temb, rotary = model.prepare(lat, enc, t, [(1, 64, 64)], [txt, txt])
    return 2 * (64 * 64 + txt) * 256 * 2, lambda: model.run_blocks(img, text, temb, rotary)


@pytest.mark.parametrize("make,option", [(_wan, False), (_wan, True), (_qwen, 64), (_qwen, 50)])
def test_native_blocks_take_no_more_memory_than_kernel_by_kernel(gpu, monkeypatch, make, option):
    peaks = []
    with torch.inference_mode():
        row, call = make(gpu, option)   # bytes of one tensor as wide as the model
        for native in (True, False):
            monkeypatch.setattr(kernels, "NATIVE_BLOCKS", native)
            call()
            torch.cuda.synchronize()
            gc.collect()  # (modules hold themselves: an earlier test's, collected during the call, would be taken off its peak)
            base = torch.cuda.memory_allocated()
            torch.cuda.reset_peak_memory_stats()
            call()
            peaks.append((torch.cuda.max_memory_allocated() - base) / row)
    print(f"{make.__name__} {option}: {peaks[0]:.2f} native, {peaks[1]:.2f} kernel by kernel (tensors of the model's width)", flush=True)
    assert peaks[0] <= peaks[1] + 0.5   # (half a tensor: text keys and values, rounding of the parts)
