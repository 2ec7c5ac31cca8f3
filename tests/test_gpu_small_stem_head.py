"""The ends of a small model in two launches: the inputs' projections with the text's norm, and the head's norm with its projection; the bits of
the launches one by one, where the kernel for small products takes those too, and a float32 sum of the same products, rounded once, in every element."""

import pytest
import torch

from vllm_omni_amd import _lib, kernels
from vllm_omni_amd.blocks.qwen_image import QwenImageTransformer2DModel
from vllm_omni_amd.layers.rmsnorm import RMSNorm

pytestmark = pytest.mark.gpu
BF16, F16 = torch.bfloat16, torch.float16


def _linear(gpu, k, n, dtype, bias=True):
    lin = torch.nn.Linear(k, n, bias=bias, device=gpu, dtype=dtype)
    with torch.no_grad():
        lin.weight.normal_(0, k ** -0.5)
    return lin


def _twice(lin, rows):
    """``lin`` of the rows [M, K] by the kernel for small products, as both problems of a pair; None where it does not take them."""
    lib, (M, K), N = _lib.load(), rows.shape, lin.out_features
    if not lib.odit_linear_pair_is_small(M, M, N, K):
        return None
    outs, q = [torch.full((M, N), float("nan"), device=rows.device, dtype=rows.dtype) for _ in range(2)], (_lib.LinearProblem * 2)()
    for p, out in zip(q, outs):
        p.x, p.w, p.bias, p.out, p.M = rows.data_ptr(), lin.weight.data_ptr(), None if lin.bias is None else lin.bias.data_ptr(), out.data_ptr(), M
        p.ldx, p.ldw, p.ldo = K, K, N
    code, epilogue = 0 if rows.dtype == BF16 else 1, _lib.ODIT_EPI_NONE if lin.bias is None else _lib.ODIT_EPI_BIAS
    # (without a workspace no other kernel runs)
    _lib.check(lib.odit_linear_pair(_lib.C.addressof(q), N, K, epilogue, 0, code, 0, None, 0, torch.cuda.current_stream().cuda_stream), "odit_linear_pair")
    assert torch.equal(*outs)
    return outs[0]


# (rows and K of both; every number of steps on either side, edges of tiles of 64)
@pytest.mark.parametrize("M0,K0,M1,K1,N", [(256, 64, 64, 256, 256), (1, 64, 1, 64, 64), (63, 192, 65, 128, 72), (128, 256, 7, 64, 520), (300, 128, 200, 256, 8), (64, 64, 64, 128, 256)])
@pytest.mark.parametrize("dtype,bias", [(BF16, True), (F16, True), (F16, False)])
def test_stem(gpu, M0, K0, M1, K1, N, dtype, bias):
    print(f"stem {M0}x{K0} {M1}x{K1} N={N} {dtype}", flush=True)
    torch.manual_seed(M0 + K1)
    a, b, norm = _linear(gpu, K0, N, dtype, bias), _linear(gpu, K1, N, dtype, bias), RMSNorm(K1).to(device=gpu, dtype=dtype)
    x = torch.randn(1, M0, K0, device=gpu).to(dtype)
    y = (torch.randn(1, M1, K1, device=gpu) * torch.randn(1, M1, 1, device=gpu).exp()).to(dtype)
    y[0, M1 // 2] = 0
    with torch.no_grad():
        norm.weight.normal_(1, 0.2)
    with torch.inference_mode():
        got = kernels.project_stem(a, x, norm, b, y)
        normed = norm(y)
        u = 2.0 ** -8 if dtype == BF16 else 2.0 ** -11
        for out, lin, rows in zip(got, (a, b), (x, normed), strict=True):
            exact, size = (torch.nn.functional.linear(f(rows.double()), f(lin.weight.double()), f(lin.bias.double()) if bias else None) for f in (lambda t: t, torch.abs))
            # the result's rounding and that of K + 1 float32 sums (an element of float16 may be below the normal numbers)
            assert bool(((out.double() - exact).abs() <= u * exact.abs() + (lin.in_features + 1) * 2.0 ** -23 * size + 2.0 ** -25).all())
            want = kernels.project(lin, rows)  # (whichever kernel takes it alone)
            assert float((out.double() - want.double()).norm()) <= (2.0 ** -9 if dtype == BF16 else 2.0 ** -12) * float(want.double().norm())
            alone = _twice(lin, rows[0])
            if alone is not None:
                assert torch.equal(out[0], alone)
        if K1 > 64 and N >= 64:  # a row at a time, in any launch, the same bits
            assert torch.equal(got[1], kernels.project_stem(a, x[:, :1], norm, b, y)[1]) and torch.equal(got[0], kernels.project_stem(a, x, norm, b, y[:, :1])[0])


@pytest.mark.parametrize("B,S,C,N", [(1, 256, 256, 64), (2, 65, 128, 136), (3, 21, 192, 128), (2, 64, 256, 72)])
@pytest.mark.parametrize("dtype", [BF16, F16])
def test_head(gpu, B, S, C, N, dtype):
    print(f"head {B}x{S}x{C} N={N} {dtype}", flush=True)
    torch.manual_seed(S)
    lin, x, head = _linear(gpu, C, N, dtype), torch.randn(B, S, C, device=gpu).to(dtype), torch.randn(B, 2 * C, device=gpu).to(dtype)
    scale, shift = head.chunk(2, dim=1)
    with torch.inference_mode():
        got = kernels.project_normed(lin, x, shift, scale, 1e-6)
        want = kernels.project(lin, kernels.adaln_modulate(x, shift, scale, eps=1e-6))
    assert torch.equal(got, want)


def test_refused(gpu):
    a, b, norm = _linear(gpu, 64, 128, BF16), _linear(gpu, 256, 128, BF16), RMSNorm(256).to(device=gpu, dtype=BF16)
    x, y = torch.randn(1, 64, 64, device=gpu, dtype=BF16), torch.randn(1, 20, 256, device=gpu, dtype=BF16)
    with torch.inference_mode():
        assert kernels.project_stem(a, x, norm, b, y) is not None
        assert kernels.project_stem(a, x.half(), norm, b, y) is None
        assert kernels.project_stem(a, x, RMSNorm(256).to(device=gpu), b, y) is None  # float32 weights
        assert kernels.project_stem(a, x, RMSNorm(192).to(device=gpu, dtype=BF16), _linear(gpu, 192, 128, BF16), y[..., :192].contiguous()) is None
        assert kernels.project_stem(a, x.repeat(1, 4096, 1), norm, b, y) is None  # too many tiles to have a place at once
        assert kernels.project_normed(a, x, x[:, 0], x[:, 1].float(), 1e-6) is None
        b.register_forward_hook(lambda *a: None)
        assert kernels.project_stem(a, x, norm, b, y) is None


def test_model(gpu, monkeypatch):
    g = torch.Generator(device=gpu).manual_seed(5)
    model = QwenImageTransformer2DModel(num_layers=2, attention_head_dim=64, num_attention_heads=4, joint_attention_dim=256, axes_dims_rope=(8, 28, 28)).to(device=gpu, dtype=BF16)
    with torch.no_grad():
        for p in model.parameters():
            p.normal_(0.0, 0.05, generator=g)
    model.fuse_modulation()
    args = dict(hidden_states=torch.randn(1, 256, 64, device=gpu, generator=g).to(BF16), encoder_hidden_states=torch.randn(1, 64, 256, device=gpu, generator=g).to(BF16),
                timestep=torch.full((1,), 0.7, device=gpu, dtype=BF16), img_shapes=[[(1, 16, 16)]], txt_seq_lens=[64], return_dict=False)
    with torch.inference_mode():
        got = model(**args)[0]
        for name in ("project_stem", "project_normed"):
            monkeypatch.setattr(kernels, name, lambda *a: None)
        assert torch.equal(got, model(**args)[0]) and bool(torch.isfinite(got).all())
