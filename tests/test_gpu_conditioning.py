"""The conditioning of a step in fewer launches: two weights on the same few rows, and a timestep's sinusoid where its first projection stages
it. Every value is one of the separate launches' bits; what the kernels do not take is refused."""

import math

import pytest
import torch

from vllm_omni_amd import _lib, kernels
from vllm_omni_amd.blocks.flux import FluxTransformer2DModel
from vllm_omni_amd.blocks.qwen_image import QwenImageTransformer2DModel, QwenTimestepProjEmbeddings, TimestepEmbedding

pytestmark = pytest.mark.gpu
BF16, F16, F32 = torch.bfloat16, torch.float16, torch.float32


def _linear(n, k, dtype, gpu, bias=True):
    lin = torch.nn.Linear(k, n, bias=bias, device=gpu, dtype=dtype)
    with torch.no_grad():
        lin.weight.normal_(0, k**-0.5)
    return lin


# K a multiple of 512 and up to 4 rows: the stream kernel (one wavefront's group must not straddle the weights); others the matrix kernel;
# the first pair of features together passes the line for four rows of W at a time
@pytest.mark.parametrize("M,N0,N1,K", [(1, 65533, 7, 512), (2, 65536, 64, 512), (2, 3, 1, 512), (4, 301, 129, 1024), (1, 1, 1, 512), (5, 33, 47, 512),
                                       (2, 24576, 512, 256), (16, 17, 15, 96), (3, 5000, 1, 32), (4, 2, 300, 3072), (8, 20000, 16, 256)])
@pytest.mark.parametrize("dtype,bias", [(BF16, True), (F16, False)])
def test_two_weights(gpu, M, N0, N1, K, dtype, bias):
    print(f"pair of few rows {M} x {N0}, {N1} x {K} {dtype}", flush=True)
    torch.manual_seed(M + N0)
    x = torch.randn(M, K + 8, device=gpu, dtype=dtype)[:, :K]
    w, lin = _linear(N0, K, dtype, gpu, bias), _linear(N1, K, dtype, gpu)
    with torch.inference_mode():
        got = kernels.linear_few_pair(x, w.weight, w.bias, lin)
        want = kernels.linear_few(x, w.weight, w.bias, silu_input=True), kernels.linear_few(x, lin.weight, lin.bias, silu_input=True)
    assert all(torch.equal(a, b) for a, b in zip(got, want, strict=True))


def test_two_weights_refused(gpu):
    x, w, lin = torch.randn(2, 64, device=gpu, dtype=BF16), torch.randn(32, 64, device=gpu, dtype=BF16), _linear(16, 64, BF16, gpu)
    with torch.inference_mode():
        assert kernels.linear_few_pair(x, w, None, lin) is not None
        assert kernels.linear_few_pair(x.half(), w, None, lin) is None  # a type of its own
        assert kernels.linear_few_pair(torch.randn(17, 64, device=gpu, dtype=BF16), w, None, lin) is None
        assert kernels.linear_few_pair(x, w[:, :32], None, lin) is None
        assert kernels.linear_few_pair(x[:, :56], w[:, :56], None, _linear(16, 56, BF16, gpu)) is None
        lin.register_forward_hook(lambda *a: None)
        assert kernels.linear_few_pair(x, w, None, lin) is None
    assert kernels.linear_few_pair(x, w, None, _linear(16, 64, BF16, gpu)) is None  # with gradients


@pytest.mark.parametrize("n", [1, 2, 5, 16])
@pytest.mark.parametrize("scale,pre,t_dtype,dtype", [(1000.0, 1.0, F32, BF16), (1000.0, 1.0, BF16, BF16), (1.0, 1000.0, F16, BF16), (1.0, 1000.0, F32, F16)])
def test_sinusoid_and_projection(gpu, n, scale, pre, t_dtype, dtype):
    print(f"time embedding {n} {scale} {pre} {t_dtype} {dtype}", flush=True)
    torch.manual_seed(n)
    for width in (256, 3072, 40):
        emb = TimestepEmbedding(256, width).to(device=gpu, dtype=dtype)
        t = torch.rand(n, device=gpu).to(t_dtype)
        with torch.inference_mode():
            got = kernels.time_embedding(emb, t, 256, 10000, scale, dtype, pre)
            rows = QwenTimestepProjEmbeddings.time_proj(t, scale=scale, dtype=dtype, pre=pre)
            if width == 40:  # no kernel of the second projection's: the module as it is
                assert got is None
                got = QwenTimestepProjEmbeddings.embed(emb, t, dtype, scale=scale, pre=pre)
            assert torch.equal(got, emb(rows))


def test_sinusoid_refused(gpu):
    emb, t = TimestepEmbedding(256, 64).to(device=gpu, dtype=BF16), torch.rand(2, device=gpu)
    assert kernels.time_embedding(emb, t, 256, 10000, 1.0, BF16) is None  # with gradients
    with torch.inference_mode():
        assert kernels.time_embedding(emb, t, 256, 10000, 1.0, BF16) is not None
        assert kernels.time_embedding(emb, t, 128, 10000, 1.0, BF16) is None
        assert kernels.time_embedding(emb, t, 256, 10000, 1.0, F16) is None
        assert kernels.time_embedding(emb, torch.rand(17, device=gpu), 256, 10000, 1.0, BF16) is None
        assert kernels.time_embedding(TimestepEmbedding(512, 64).to(device=gpu, dtype=BF16), t, 512, 10000, 1.0, BF16) is None  # another order of summation
    lib, w, out = _lib.load(), emb.linear_1.weight, torch.zeros(2, 64, device=gpu, dtype=BF16)
    call = [t.data_ptr(), w.data_ptr(), None, out.data_ptr(), 2, 64, 256, 256, 64, -math.log(10000), 1.0, 1.0, _lib.ODIT_F32, _lib.ODIT_BF16, None]
    for at, value, code in ((0, None, -1), (5, 0, -1), (7, 255, -1), (8, 63, -1), (6, 248, -2), (4, 17, -2), (13, _lib.ODIT_F32, -2)):
        assert lib.odit_time_linear(*call[:at], value, *call[at + 1:]) == code, at


@pytest.mark.parametrize("flux", [False, True])
@pytest.mark.parametrize("B", [1, 3])
def test_models(gpu, monkeypatch, flux, B):
    print(f"conditioning of a model, flux={flux} B={B}", flush=True)
    g = torch.Generator(device=gpu).manual_seed(7)
    common = dict(num_layers=2, attention_head_dim=64, num_attention_heads=4, joint_attention_dim=256, axes_dims_rope=(8, 28, 28))
    model = (FluxTransformer2DModel(num_single_layers=1, pooled_projection_dim=128, **common) if flux
             else QwenImageTransformer2DModel(**common)).to(device=gpu, dtype=BF16)
    with torch.no_grad():
        for p in model.parameters():
            p.normal_(0.0, 0.05, generator=g)
    model.fuse_modulation()
    rand = lambda *s: torch.randn(*s, device=gpu, generator=g).to(BF16)  # noqa: E731
    args = dict(hidden_states=rand(B, 48, 64), encoder_hidden_states=rand(B, 9, 256), timestep=torch.full((B,), 0.7, device=gpu, dtype=BF16),
                return_dict=False)
    if flux:
        args |= dict(pooled_projections=rand(B, 128), guidance=torch.full((B,), 3.5, device=gpu), img_ids=torch.zeros(48, 3, device=gpu),
                     txt_ids=torch.zeros(9, 3, device=gpu))
    else:
        args |= dict(img_shapes=[[(1, 6, 8)]] * B, txt_seq_lens=[9] * B)
    with torch.inference_mode():
        got = model(**args)[0]
        calls = []
        monkeypatch.setattr(model, "finish", lambda *a, **k: calls.append(k) or type(model).finish(model, *a, **k))
        assert torch.equal(model(**args)[0], got) and calls == [{"return_dict": False}]  # a stage of one's own is called as ever
        for name in ("linear_few_pair", "time_embedding"):
            monkeypatch.setattr(kernels, name, lambda *a, **k: None)
        want = model(**args)[0]
    assert bool(torch.isfinite(want).all()) and torch.equal(got, want)
