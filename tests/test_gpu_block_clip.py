"""Blocks in float16 whose results pass the largest finite value: both streams of a Qwen-Image block, the text's of a dual Flux block and a single Flux block clip theirs, the
image stream of a dual Flux block does not (qwen_image_transformer.py:809-815, flux_transformer.py:310-314, 362-364). One native call, whose last projections clip on their way or
leave it to a pass, against the same block through the per-kernel wrappers, which clip behind it; by every route that a gated projection has."""

import pytest
import torch

from vllm_omni_amd import kernels
from vllm_omni_amd.blocks.flux import FluxRotary, FluxSingleTransformerBlock, FluxTransformerBlock
from vllm_omni_amd.blocks.qwen_image import QwenImageTransformerBlock

pytestmark = pytest.mark.gpu

MOST = 65504.0


@pytest.fixture(params=["auto", "library", "handwritten"])
def engine(request):
    kernels.set_linear_engine(request.param)
    yield request.param
    kernels.set_linear_engine("auto")


def _made(block, gpu, g):
    block = block.to(device=gpu, dtype=torch.half).eval().requires_grad_(False)
    for name, p in block.named_parameters():
        p.normal_(1.0 if "norm" in name and name.endswith("weight") and p.dim() == 1 else 0.0, 0.03, generator=g)
    return block


def _stream(gpu, g, B, S, C):
    """Rows whose features are near either limit, but for every third."""
    x = torch.randn(B, S, C, device=gpu, generator=g).sign() * 65500
    x[..., ::3] = torch.randn(B, S, (C + 2) // 3, device=gpu, generator=g)
    return x.half()


def _mods(gpu, g, B, C, parts):
    """shift, scale, gate, `parts` times: the last gate takes results over the limit, the first (of the attention, whose rows are normed again) does not."""
    m = 0.1 * torch.randn(B, parts, 3, C, device=gpu, generator=g)
    m[:, :, 2] *= 0.01
    m[:, -1, 2] = 60 * torch.randn(B, C, device=gpu, generator=g)
    return m.flatten(1).half()


def _gate_rows(mods, biases, parts):
    """float32 gates and gates times biases, [B, streams, parts, C]"""
    C = mods[0].shape[1] // (3 * parts)
    gates = torch.stack([m.view(m.shape[0], parts, 3, C)[:, :, 2].float() for m in mods], dim=1)
    return gates, gates * torch.stack([torch.stack([b.float() for b in s]) for s in biases])[None]


def _runs(monkeypatch, call):
    """(results of one native call, of the wrappers)"""
    with torch.inference_mode():
        with monkeypatch.context() as m:  # (what goes through a wrapper is not one native call)
            m.setattr(kernels, "linear", None)
            native = call()
        with monkeypatch.context() as m:
            m.setattr(kernels, "NATIVE_BLOCKS", False)
            stepwise = call()
    return native, stepwise


def _same(got, want, clipped, halves=False):
    assert not bool(got.isnan().any()) and not bool(want.isnan().any())
    if clipped:
        assert float(got.abs().max()) == MOST
        assert float((got.abs() == MOST).float().mean()) > 0.05, "results past the limit"
    else:
        assert float(got.isinf().float().mean()) > 0.05, "results past the limit, as they come"
    # Two orders of summation: a rounding of the result, and 2^-8 (a rounding each of the rows, the hidden ones and attention's) of what the gated
    # projection adds (at most about 6 sigma, 6 * 60). A result on the one side of the limit and infinite on the other: one spacing, 32.
    # `halves`: the wrappers add two products one after the other; the sum after the first is rounded (16 at most), and where it is infinite it stays so whatever the
    # second takes off again (6 sigma of its gate, 6 * 60).
    a, b = (t.double().clamp(-65536, 65536) for t in (got, want))
    bound = 2.0 ** -10 * b.abs() + 2.0 ** -8 * 360 + (0 if clipped else 32)
    if halves:
        bound += torch.where(b.abs() == MOST, 360.0, 16.0)
    assert bool(((a - b).abs() <= bound).all()), float((a - b).abs().max())


# rows of a few tiles of the small kernel; of the stream-K and the tile kernel; entries whose gates change inside a tile; few and many enough for the library's gated form
@pytest.mark.parametrize("B, S_img, S_txt, H, D", [(1, 70, 20, 4, 64), (2, 70, 20, 4, 64), (1, 700, 300, 8, 128), (2, 330, 90, 8, 128), (2, 1100, 33, 8, 128), (1, 1300, 140, 24, 128)])
@pytest.mark.parametrize("rows", [False, True])
def test_qwen_image(gpu, monkeypatch, engine, B, S_img, S_txt, H, D, rows):
    g, C = torch.Generator(device=gpu).manual_seed(S_img), H * D
    block = _made(QwenImageTransformerBlock(C, H, D), gpu, g)
    mods = [_mods(gpu, g, B, C, 2) for _ in range(2)]
    gate_rows = _gate_rows(mods, [[block.attn.to_out.bias, block.img_mlp.net[2].bias], [block.attn.to_add_out.bias, block.txt_mlp.net[2].bias]], 2) if rows else None
    img, txt = _stream(gpu, g, B, S_img, C), _stream(gpu, g, B, S_txt, C)
    freqs = [torch.polar(torch.ones(S, D // 2, device=gpu), 6 * torch.rand(S, D // 2, device=gpu, generator=g)) for S in (S_img, S_txt)]
    print(f"clip in a block B={B} {S_img}+{S_txt} C={C} {engine} rows={rows}", flush=True)
    native, stepwise = _runs(monkeypatch, lambda: block(img, txt, None, None, freqs, mod_params=tuple(mods), gate_rows=gate_rows))
    for got, want in zip(native, stepwise):
        _same(got, want, True)


@pytest.mark.parametrize("B", [1, 2])
def test_qwen_image_with_a_modulation_per_token(gpu, monkeypatch, engine, B):
    g, S_img, S_txt, H, D = torch.Generator(device=gpu).manual_seed(B), 330, 40, 8, 128
    C = H * D
    block = _made(QwenImageTransformerBlock(C, H, D, zero_cond_t=True), gpu, g)
    mods = (_mods(gpu, g, 2 * B, C, 2), _mods(gpu, g, B, C, 2))
    index = torch.randint(0, 2, (B, S_img), device=gpu, generator=g).int()
    img, txt = _stream(gpu, g, B, S_img, C), _stream(gpu, g, B, S_txt, C)
    freqs = [torch.polar(torch.ones(S, D // 2, device=gpu), 6 * torch.rand(S, D // 2, device=gpu, generator=g)) for S in (S_img, S_txt)]
    print(f"clip in a block, modulation per token B={B} {engine}", flush=True)
    native, stepwise = _runs(monkeypatch, lambda: block(img, txt, None, None, freqs, mod_params=mods, modulate_index=index))
    for got, want in zip(native, stepwise):
        _same(got, want, True)


def _rotary(gpu, g, S, D):
    a = 6 * torch.rand(S, D // 2, device=gpu, generator=g)
    return FluxRotary(a.cos(), a.sin())


@pytest.mark.parametrize("B, S_img, S_txt, H, D", [(1, 70, 20, 4, 64), (2, 330, 90, 8, 128), (1, 1300, 140, 24, 128)])
@pytest.mark.parametrize("rows", [False, True])
def test_flux_dual(gpu, monkeypatch, engine, B, S_img, S_txt, H, D, rows):
    g, C = torch.Generator(device=gpu).manual_seed(S_img), H * D
    block = _made(FluxTransformerBlock(C, H, D), gpu, g)
    mods = [_mods(gpu, g, B, C, 2) for _ in range(2)]
    gate_rows = _gate_rows(mods, [[block.attn.to_out[0].bias, block.ff.net[2].bias], [block.attn.to_add_out.bias, block.ff_context.net[2].bias]], 2) if rows else None
    img, txt, rot = _stream(gpu, g, B, S_img, C), _stream(gpu, g, B, S_txt, C), _rotary(gpu, g, S_img + S_txt, D)
    print(f"clip in a dual block B={B} {S_img}+{S_txt} C={C} {engine} rows={rows}", flush=True)
    native, stepwise = _runs(monkeypatch, lambda: block(img, txt, None, rot, mod_params=tuple(mods), gate_rows=gate_rows))
    _same(native[0], stepwise[0], True)
    _same(native[1], stepwise[1], False)


# two products that add up (few rows, and by the library), and one over both tensors
@pytest.mark.parametrize("B, S, H, D", [(1, 90, 4, 64), (2, 330, 8, 128), (1, 1440, 24, 128)])
@pytest.mark.parametrize("in_place", [False, True])
def test_flux_single(gpu, monkeypatch, engine, B, S, H, D, in_place):
    g, C = torch.Generator(device=gpu).manual_seed(S), H * D
    block = _made(FluxSingleTransformerBlock(C, H, D), gpu, g)
    mod = _mods(gpu, g, B, C, 1)
    gate = mod[:, 2 * C:].float()
    x, rot = _stream(gpu, g, B, S, C), _rotary(gpu, g, S, D)
    print(f"clip in a single block B={B} S={S} C={C} {engine}", flush=True)
    native, stepwise = _runs(monkeypatch, lambda: block.forward_joint(x.clone(), None, rot, mod=mod, in_place=in_place, gate_rows=(gate, gate * block.proj_out.bias.float())))
    _same(native, stepwise, True, halves=True)
