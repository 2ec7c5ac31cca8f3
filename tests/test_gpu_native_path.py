"""The native host path (csrc/native.cpp): a block as one native call against the same block through the per-kernel
wrappers, whose results the oracle tests pin, and module trees it has to leave alone."""

import pytest
import torch

pytestmark = pytest.mark.gpu


def _init(model, gpu, dtype):
    g = torch.Generator().manual_seed(0)
    for name, p in model.named_parameters():
        v = torch.randn(p.shape, generator=g) * 0.02
        p.data = (v + 1 if "norm" in name and name.endswith("weight") and p.dim() == 1 else v).to(gpu).to(dtype)
    return model.eval()


def _qwen(gpu, dtype, txt, masked):
    from vllm_omni_amd.blocks.qwen_image import QwenImageTransformer2DModel

    model = _init(QwenImageTransformer2DModel(num_layers=2, attention_head_dim=64, num_attention_heads=4, joint_attention_dim=256,
                                              axes_dims_rope=(8, 28, 28)), gpu, dtype)
    model.fuse_modulation()
    g = torch.Generator().manual_seed(1)
    lat, enc = torch.randn(2, 63, 64, generator=g).to(dtype).to(gpu), torch.randn(2, txt, 256, generator=g).to(dtype).to(gpu)
    mask = None
    if masked:
        mask = torch.ones(2, txt, dtype=torch.bool)
        mask[1, txt // 2:] = False
        mask = mask.to(gpu)
    t = torch.tensor([0.3, 0.3]).to(dtype).to(gpu)
    return model, lambda: model(lat, enc, mask, t, [(1, 7, 9)], [txt, txt]).sample


def _qwen_edit(gpu, dtype, txt, _):
    """The editing variant: two images, a conditioning choice per token."""
    from vllm_omni_amd.blocks.qwen_image import QwenImageTransformer2DModel

    model = _init(QwenImageTransformer2DModel(num_layers=2, attention_head_dim=64, num_attention_heads=4, joint_attention_dim=256,
                                              axes_dims_rope=(8, 28, 28), zero_cond_t=True), gpu, dtype)
    model.fuse_modulation()
    g = torch.Generator().manual_seed(4)
    lat, enc = torch.randn(2, 63 + 20, 64, generator=g).to(dtype).to(gpu), torch.randn(2, txt, 256, generator=g).to(dtype).to(gpu)
    t = torch.tensor([0.3, 0.3]).to(dtype).to(gpu)
    return model, lambda: model(lat, enc, None, t, [[(1, 7, 9), (1, 4, 5)]] * 2, [txt, txt]).sample


def _flux(gpu, dtype, txt, masked):
    from vllm_omni_amd.blocks.flux import FluxTransformer2DModel

    model = _init(FluxTransformer2DModel(num_layers=1, num_single_layers=2, attention_head_dim=64, num_attention_heads=4,
                                         joint_attention_dim=256, pooled_projection_dim=64, axes_dims_rope=(8, 28, 28)), gpu, dtype)
    model.fuse_modulation()
    g = torch.Generator().manual_seed(2)
    lat, enc = torch.randn(1, 63, 64, generator=g).to(dtype).to(gpu), torch.randn(1, txt, 256, generator=g).to(dtype).to(gpu)
    pooled = torch.randn(1, 64, generator=g).to(dtype).to(gpu)
    ids = torch.randint(0, 9, (63, 3), generator=g).float().to(gpu)
    one = torch.ones(1, device=gpu)
    return model, lambda: model(lat, enc, pooled, 0.3 * one, ids, torch.zeros(txt, 3, device=gpu), 3.5 * one).sample


def _wan(gpu, dtype, txt, per_token):
    from vllm_omni_amd.blocks.wan import WanTransformer3DModel

    model = _init(WanTransformer3DModel(num_attention_heads=4, attention_head_dim=64, text_dim=128, ffn_dim=512, num_layers=2), gpu, dtype)
    g = torch.Generator().manual_seed(3)
    video, text = torch.randn(2, 16, 3, 6, 14, generator=g).to(dtype).to(gpu), torch.randn(2, txt, 128, generator=g).to(dtype).to(gpu)
    t = torch.randint(1, 999, (2, 63) if per_token else (2,), generator=g).float().to(gpu)
    return model, lambda: model(video, t, text).sample


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("make,txt,option", [(_qwen, 64, False), (_qwen, 19, True), (_qwen_edit, 19, False), (_flux, 64, False), (_flux, 7, False),
                                             (_wan, 13, False), (_wan, 13, True)])
def test_native_block_equals_the_per_kernel_path(gpu, monkeypatch, dtype, make, txt, option):
    from vllm_omni_amd import kernels

    model, call = make(gpu, dtype, txt, option)
    with torch.inference_mode():
        native = call()
        monkeypatch.setattr(kernels, "NATIVE_BLOCKS", False)
        stepwise = call()
    print(f"native block {make.__name__} {dtype}: max diff {(native - stepwise).abs().max().item():.2e}", flush=True)
    tol = 2e-2 if dtype == torch.bfloat16 else 3e-3
    torch.testing.assert_close(native.float(), stepwise.float(), atol=tol, rtol=tol)


def test_native_block_leaves_changed_modules_to_python(gpu, monkeypatch):
    """A hook on a projection runs, and a replaced projection is the one that is used."""
    from vllm_omni_amd import kernels

    class Doubled(torch.nn.Linear):
        def forward(self, x):
            return 2 * super().forward(x)

    model, call = _qwen(gpu, torch.bfloat16, 64, False)
    attn = model.transformer_blocks[0].attn
    with torch.inference_mode():
        plain = call()
        seen = []
        handle = attn.to_qkv.register_forward_hook(lambda *a: seen.append(1))
        hooked = call()
        handle.remove()
    assert seen == [1]
    torch.testing.assert_close(hooked.float(), plain.float(), atol=2e-2, rtol=2e-2)
    new = Doubled(attn.to_qkv.in_features, attn.to_qkv.out_features, device=gpu, dtype=torch.bfloat16)
    new.load_state_dict(attn.to_qkv.state_dict())
    attn.to_qkv = new
    with torch.inference_mode():
        changed = call()
        monkeypatch.setattr(kernels, "NATIVE_BLOCKS", False)
        stepwise = call()
    torch.testing.assert_close(changed.float(), stepwise.float(), atol=2e-2, rtol=2e-2)
    assert (changed - plain).float().norm() > 2 * (changed - stepwise).float().norm()
