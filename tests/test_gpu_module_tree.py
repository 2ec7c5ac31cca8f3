"""What a user changes in a module tree takes effect: hooks run, replaced submodules and switches are used, although a
plain tree runs through native calls that never call the modules."""

import pytest
import torch

from test_gpu_native_path import _flux, _qwen, _wan
from vllm_omni_amd.hooks.base import HookRegistry, ModelHook

pytestmark = pytest.mark.gpu


def _both(monkeypatch, call):
    """(result of the default path, result of the per-kernel path)"""
    from vllm_omni_amd import kernels

    with torch.inference_mode():
        native = call()
        with monkeypatch.context() as m:
            m.setattr(kernels, "NATIVE_BLOCKS", False)
            stepwise = call()
    return native.float(), stepwise.float()


def _single_norm(model):
    return model.single_transformer_blocks[0].norm


def test_hook_and_replaced_norm_of_a_flux_single_block(gpu, monkeypatch):
    from vllm_omni_amd.blocks.flux import AdaLayerNormZeroSingle

    class Scaled(AdaLayerNormZeroSingle):
        def forward(self, x, emb=None, mod=None):
            n, gate = super().forward(x, emb, mod)
            return 3 * n, gate

    model, call = _flux(gpu, torch.bfloat16, 64, False)
    plain, _ = _both(monkeypatch, call)
    seen = []
    handle = _single_norm(model).register_forward_hook(lambda *a: seen.append(1))
    with torch.inference_mode():
        call()
        handle.remove()

        class Count(ModelHook):
            def pre_forward(self, module, *args, **kwargs):
                seen.append(2)
                return args, kwargs

        HookRegistry.get_or_create(_single_norm(model)).register_hook("count", Count())
        call()
    assert seen == [1, 2]
    new = Scaled(256).to(gpu).to(torch.bfloat16)
    new.load_state_dict({k: v for k, v in _single_norm(model).state_dict().items()})
    model.single_transformer_blocks[0].norm = new
    native, stepwise = _both(monkeypatch, call)
    torch.testing.assert_close(native, stepwise, atol=2e-2, rtol=2e-2)
    assert (native - plain).norm() > 2 * (native - stepwise).norm()


def _attention_scale(model, block):
    block.attn.attn.attention.softmax_scale *= 4


def _qk_ref_rounding(model, block):
    block.attn.ref_rounding = True


def _unfused_mlp(model, block):
    (block.img_mlp if hasattr(block, "img_mlp") else block.ff).net[0].fused = False


@pytest.mark.parametrize("change", [_attention_scale, _qk_ref_rounding, _unfused_mlp])
@pytest.mark.parametrize("make", [_qwen, _flux])
def test_switches_on_submodules_are_read(gpu, monkeypatch, make, change):
    """A switch set on one submodule sends its block to Python (the same bits as without the native path); a scale set on
    the attention's backend object is the one that the native block uses."""
    model, call = make(gpu, torch.bfloat16, 64, False)
    out = []
    model.transformer_blocks[-1].register_forward_hook(lambda m, a, result: out.append(torch.cat(result, dim=1).float()))
    _both(monkeypatch, call)
    for block in model.transformer_blocks:
        change(model, block)
    _both(monkeypatch, call)
    plain, _, native, stepwise = out
    if change is _attention_scale:
        torch.testing.assert_close(native, stepwise, atol=2e-2, rtol=2e-2)
        assert (native - plain).norm() > 2 * (native - stepwise).norm()
    else:
        assert torch.equal(native, stepwise)


def test_position_embedders_are_called_unless_plain(gpu):
    """A subclass with its own positions is used, hooks run, and a module with nothing but ``forward`` is enough."""
    from vllm_omni_amd.blocks.flux import FluxPosEmbed
    from vllm_omni_amd.blocks.qwen_image import QwenEmbedRope

    class HalfFlux(FluxPosEmbed):
        def forward(self, ids):
            return super().forward(ids * 0.5)

    class OnlyForward(torch.nn.Module):
        def __init__(self, inner):
            super().__init__()
            self.inner = inner

        def forward(self, *args, **kwargs):
            return tuple(self.inner(*args, **kwargs))

    class NearerText(QwenEmbedRope):
        def forward(self, video_fhw, txt_seq_lens, device):
            vid, txt = super().forward(video_fhw, txt_seq_lens, device)
            return vid, txt * txt

    for make, cls, own in ((_flux, HalfFlux, lambda: HalfFlux(10000, [8, 28, 28])),
                           (_qwen, NearerText, lambda: NearerText(10000, [8, 28, 28]))):
        model, call = make(gpu, torch.bfloat16, 64, False)
        seen = []
        with torch.inference_mode():
            plain = call()
            handle = model.pos_embed.register_forward_hook(lambda *a: seen.append(1))
            hooked = call()
            handle.remove()
            model.pos_embed = OnlyForward(model.pos_embed)
            wrapped = call()
            model.pos_embed = own()
            changed = call()
        assert seen == [1]
        # (the float32 tables are made another way: from float64 or from complex ones)
        torch.testing.assert_close(hooked.float(), plain.float(), atol=2e-2, rtol=2e-2)
        assert torch.equal(wrapped, hooked)
        assert (changed - plain).float().norm() > 2 * (hooked - plain).float().norm() and not torch.equal(changed, plain)


def test_wrapped_time_embedding_gets_the_scaled_timestep(gpu):
    model, call = _flux(gpu, torch.bfloat16, 64, False)
    inner, seen = model.time_text_embed.forward, []

    def forward(timestep, guidance, pooled):   # an offloading wrapper of the documented signature
        seen.append(timestep.item())
        return inner(timestep, guidance, pooled)

    with torch.inference_mode():
        plain = call()
        model.time_text_embed.forward = forward
        wrapped = call()
    assert seen == [torch.tensor(0.3).bfloat16().mul(1000).item()]
    assert torch.equal(plain, wrapped)


@pytest.mark.parametrize("make,option", [(_qwen, False), (_flux, False), (_wan, False), (_wan, True)])
def test_parameters_written_through_data_are_used(gpu, monkeypatch, make, option):
    """As a weight loader writes them, without a trace in version counters or addresses: the second forward is that of the
    new values, on both paths."""
    model, call = make(gpu, torch.bfloat16, 64, option)
    before, _ = _both(monkeypatch, call)
    g = torch.Generator(device=gpu).manual_seed(7)
    for name, p in model.named_parameters():
        if name.endswith("bias") or "norm" in name or "scale_shift_table" in name:
            p.data.copy_(p + 0.3 * torch.randn(p.shape, device=gpu, generator=g).to(p.dtype))
    native, stepwise = _both(monkeypatch, call)
    bound = 2.0 ** -5   # both paths round at every operation (2^-9); the new values move the result by far more
    assert (native - stepwise).norm() <= bound * stepwise.norm()
    assert (native - before).norm() > 4 * bound * before.norm()


def test_projection_with_a_hook_or_of_another_class_at_sizes_of_the_hand_written_kernels(gpu):
    """What ``project`` hands to a hand-written GEMM is the projection of a plain Linear only (1536 x 9216 x 3072 goes to the tile kernel)."""
    from vllm_omni_amd import kernels
    from vllm_omni_amd.blocks.qwen_image import project

    class Doubled(torch.nn.Linear):
        def forward(self, x):
            return 2 * super().forward(x)

    M, N, K = 1536, 9216, 3072
    g = torch.Generator(device=gpu).manual_seed(0)
    x = torch.randn(M, K, device=gpu, generator=g).bfloat16()
    lin, other = (cls(K, N, device=gpu, dtype=torch.bfloat16) for cls in (torch.nn.Linear, Doubled))
    other.load_state_dict(lin.state_dict())
    with torch.inference_mode():
        assert kernels.linear(x, lin.weight, lin.bias, plan_only=True)[0]
        plain = project(lin, x)
        seen = []
        handle = lin.register_forward_hook(lambda *a: seen.append(1))
        hooked = project(lin, x)
        handle.remove()
        assert seen == [1]
        assert ((hooked - plain).float().norm() / plain.float().norm()).item() < 2.0 ** -8
        assert ((project(other, x) - 2 * plain).float().norm() / plain.float().norm()).item() < 2.0 ** -7
