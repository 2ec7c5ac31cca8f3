"""The one-launch kernels around the transformer in a denoise step against the torch expressions they replace."""

import math

import pytest
import torch

from vllm_omni_amd import kernels

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("shape", [(1, 1, 8), (1, 31, 64), (1, 33, 136), (1, 4097, 64), (1, 16, 3, 5, 41)])
@torch.inference_mode()
def test_cfg_combine_and_euler(shape, dtype):
    pos, neg, x = (torch.randn(shape, device="cuda").to(dtype) for _ in range(3))
    comb = neg + 4.0 * (pos - neg)
    assert torch.equal(kernels.cfg_combine(pos, neg, 4.0, False), comb)
    out = kernels.cfg_combine(pos, neg, 4.0, True)
    if shape[-1] % 8:
        assert out is None
    else:  # the sums of squares are added in another order: a rounding of the norm may differ
        want = comb * (torch.norm(pos, dim=-1, keepdim=True) / torch.norm(comb, dim=-1, keepdim=True))
        torch.testing.assert_close(out, want, rtol=2e-2 if dtype == torch.bfloat16 else 2e-3, atol=1e-6)
    dt = 0.66 - 0.7
    assert torch.equal(kernels.euler_step(x, pos, dt), (x.float() + dt * pos.float()).to(dtype))


@pytest.mark.parametrize("t_dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("n,dim,scale", [(1, 256, 1000.0), (7, 256, 1.0), (5000, 64, 1.0), (3, 6, 1.0)])
@torch.inference_mode()
def test_time_sinusoid(n, dim, scale, t_dtype):
    t = (torch.rand(n, device="cuda") * 1000.0 / scale).to(t_dtype)
    half = dim // 2
    freqs = torch.exp(-math.log(10000) * torch.arange(half, dtype=torch.float32, device="cuda") / half)
    arg = scale * (t[:, None].float() * freqs[None, :])
    want = torch.cat((torch.cos(arg), torch.sin(arg)), dim=-1)
    out = kernels.time_sinusoid(t, dim, 10000, scale, torch.float32)
    torch.testing.assert_close(out, want, rtol=0, atol=2e-4)
    assert torch.equal(kernels.time_sinusoid(t, dim, 10000, scale, torch.bfloat16), out.to(torch.bfloat16))
    pre = kernels.time_sinusoid(t, dim, 10000, scale, torch.bfloat16, 1000.0)
    scaled = (t.to(torch.bfloat16) * 1000).float()
    assert torch.equal(pre, kernels.time_sinusoid(scaled, dim, 10000, scale, torch.bfloat16))


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("axes", [(16, 56, 56), (8, 28, 28), (32, 80, 80)])
@pytest.mark.parametrize("n_txt,n_img", [(0, 1), (1, 0), (7, 8), (15, 2), (512, 1025)])
@torch.inference_mode()
def test_rope_tables(n_txt, n_img, axes, dtype):
    from vllm_omni_amd.blocks.flux import FluxPosEmbed
    txt, img = ((torch.rand(n, 3, device="cuda") * 200).round().to(dtype) for n in (n_txt, n_img))
    cos, sin = kernels.rope_tables(txt, img, axes, 10000)
    want = FluxPosEmbed(10000, list(axes))(torch.cat((txt, img)).cpu())
    torch.testing.assert_close(cos.cpu(), want[0].float(), rtol=0, atol=1e-7)
    torch.testing.assert_close(sin.cpu(), want[1].float(), rtol=0, atol=1e-7)
