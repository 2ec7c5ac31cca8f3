"""One native block of each kind at the width its model has, with few and ragged rows, against the same block kernel by kernel."""

import pytest
import torch

from vllm_omni_amd import kernels

pytestmark = pytest.mark.gpu


def _fill(model, dtype, seed=0):
    g = torch.Generator(device="cuda").manual_seed(seed)
    model = model.to(dtype)
    for name, p in model.named_parameters():
        v = torch.randn(p.shape, device="cuda", generator=g) * 0.02
        p.data = (v + 1 if "norm" in name and name.endswith("weight") and p.dim() == 1 else v).to(dtype)
    return model.eval()


def _built(cls, dtype, **kw):
    with torch.device("cuda"):
        return _fill(cls(**kw), dtype)


def _rand(dtype, *shape):
    return torch.randn(shape, device="cuda", generator=torch.Generator(device="cuda").manual_seed(sum(shape))).to(dtype)


def _qwen(dtype):
    from vllm_omni_amd.blocks.qwen_image import QwenImageTransformer2DModel

    model = _built(QwenImageTransformer2DModel, dtype, num_layers=1, joint_attention_dim=256)
    model.fuse_modulation()
    mask = torch.ones(2, 71, dtype=torch.bool, device="cuda")
    mask[1, 33:] = False
    t = torch.full((2,), 0.4, device="cuda").to(dtype)
    return lambda: model(_rand(dtype, 2, 13 * 17, 64), _rand(dtype, 2, 71, 256), mask, t, [(1, 13, 17)], [71, 71]).sample


def _flux(dtype):
    from vllm_omni_amd.blocks.flux import FluxTransformer2DModel

    model = _built(FluxTransformer2DModel, dtype, num_layers=1, num_single_layers=1, joint_attention_dim=256, pooled_projection_dim=64)
    model.fuse_modulation()
    ids = torch.zeros(13 * 17, 3, device="cuda")
    ids[:, 1], ids[:, 2] = torch.arange(13 * 17) // 17, torch.arange(13 * 17) % 17
    one = torch.ones(1, device="cuda")
    return lambda: model(_rand(dtype, 1, 13 * 17, 64), _rand(dtype, 1, 71, 256), _rand(dtype, 1, 64), 0.3 * one, ids,
                         torch.zeros(71, 3, device="cuda"), 3.5 * one).sample


def _wan(dtype):
    from vllm_omni_amd.blocks.wan import WanTransformer3DModel

    model = _built(WanTransformer3DModel, dtype, num_layers=1, text_dim=128)
    t = torch.full((2,), 500.0, device="cuda")
    return lambda: model(_rand(dtype, 2, 16, 3, 14, 22), t, _rand(dtype, 2, 71, 128)).sample


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("make", [_qwen, _flux, _wan])
def test_native_block_at_model_width(gpu, monkeypatch, make, dtype):
    with torch.inference_mode():
        call = make(dtype)
        native = call().float()
        monkeypatch.setattr(kernels, "NATIVE_BLOCKS", False)
        stepwise = call().float()
    err = ((native - stepwise).norm() / stepwise.norm()).item()
    print(f"{make.__name__} {dtype}: relative difference {err:.2e}", flush=True)
    # sums in another order round to a neighbour of the type now and then, at each of a block's dozen roundings: half a step
    # (2^-9 and 2^-12 of the value) each, adding up like random ones
    assert err <= 12 ** 0.5 * (2.0 ** -9 if dtype == torch.bfloat16 else 2.0 ** -12)
