"""A step's embedders of timestep, guidance and pooled text in two launches: the bits of each by itself and of the sums, and what is refused."""

import pytest
import torch

from vllm_omni_amd import kernels
from vllm_omni_amd.blocks.flux import CombinedTimestepGuidanceTextProjEmbeddings
from vllm_omni_amd.blocks.qwen_image import QwenTimestepProjEmbeddings

pytestmark = pytest.mark.gpu
BF16, F16, F32 = torch.bfloat16, torch.float16, torch.float32


def _embedders(gpu, N, K, dtype, guided=True, bias=True):
    torch.manual_seed(N + K)
    m = CombinedTimestepGuidanceTextProjEmbeddings(N, K, guided).to(device=gpu, dtype=dtype)
    if not bias:
        m.text_embedder.linear_1.bias = m.timestep_embedder.linear_2.bias = None
    return m


def _together(m, t, guidance, pooled, pre):
    return kernels.embed_sum(m.timestep_embedder, t, None if guidance is None else m.guidance_embedder, guidance, m.text_embedder, pooled, 256, 10000, 1.0, pre)


def _apart(m, t, guidance, pooled, pre):
    rows = lambda x: QwenTimestepProjEmbeddings.time_proj(x, scale=1.0, dtype=pooled.dtype, pre=pre)  # noqa: E731
    emb = m.timestep_embedder(rows(t))
    if guidance is not None:
        emb = emb + m.guidance_embedder(rows(guidance))
    return emb + m.text_embedder(pooled)


# one, two and four rows of the second projections' kernel; chunks of the reduction: one, an odd and an even number; a text narrower and wider than the sinusoid
@pytest.mark.parametrize("M,N,K", [(1, 512, 32), (1, 1536, 768), (2, 3072, 768), (3, 512, 96), (4, 3072, 768), (4, 1024, 2080), (1, 5120, 288)])
@pytest.mark.parametrize("dtype,t_dtype,guided,bias", [(BF16, BF16, True, True), (F16, F32, True, False), (BF16, F16, False, True)])
def test_bits_of_the_separate_launches(gpu, M, N, K, dtype, t_dtype, guided, bias):
    print(f"embedders M={M} N={N} K={K} {dtype} {t_dtype} guided={guided}", flush=True)
    m = _embedders(gpu, N, K, dtype, guided, bias)
    t, pooled = torch.rand(M, device=gpu).to(t_dtype), torch.randn(M, K + 8, device=gpu).to(dtype)[:, :K]
    guidance = torch.rand(M, device=gpu) * 5 if guided else None
    with torch.inference_mode():
        for pre in (1000.0, 1.0):
            got = _together(m, t, guidance, pooled, pre)
            want = _apart(m, t, guidance, pooled, pre)
            assert got is not None and torch.equal(got, want) and torch.equal(m(t, guidance, pooled, pre=pre), want)


def test_what_is_left_to_the_separate_launches(gpu):
    rand = lambda *s: torch.randn(*s, device=gpu).to(BF16)  # noqa: E731
    with torch.inference_mode():
        for N, K, M in ((512, 512, 1), (1024, 48, 1), (520, 96, 2), (512, 96, 5), (15872, 96, 4)):  # another order of summation, steps of 32, of 512, rows, LDS
            m, t, pooled = _embedders(gpu, N, K, BF16), torch.rand(M, device=gpu), rand(M, K)
            assert _together(m, t, t, pooled, 1000.0) is None
            assert torch.equal(m(t, t, pooled, pre=1000.0), _apart(m, t, t, pooled, 1000.0))
        m, t, pooled = _embedders(gpu, 512, 96, BF16), torch.rand(2, device=gpu), rand(2, 96)
        assert _together(m, t, t, pooled, 1.0) is not None
        assert _together(m, t[:1], t, pooled, 1.0) is None and _together(m, t, t[:1], pooled, 1.0) is None  # rows that would be repeated
        assert _together(m, t, t, pooled.float(), 1.0) is None and _together(m, t, t, rand(2, 2, 96)[:, 0, ::1].t().contiguous().t(), 1.0) is None
        m.guidance_embedder.linear_2.register_forward_hook(lambda mod, a, out: out + 1)
        assert _together(m, t, t, pooled, 1.0) is None and torch.equal(m(t, t, pooled), _apart(m, t, t, pooled, 1.0))
    m = _embedders(gpu, 512, 96, BF16)
    assert _together(m, t, t, pooled, 1.0) is None  # with gradients


def test_replaced_methods_are_called(gpu, monkeypatch):
    """What a program has put on a class, as on a module, takes effect."""
    from vllm_omni_amd.blocks.flux import PixArtAlphaTextProjection

    m, t, pooled = _embedders(gpu, 512, 96, BF16), torch.rand(2, device=gpu), torch.randn(2, 96, device=gpu).to(BF16)
    with torch.inference_mode():
        text, times = m.text_embedder(pooled), QwenTimestepProjEmbeddings.embed(m.timestep_embedder, t, BF16, scale=1.0)
        with monkeypatch.context() as p:
            p.setattr(PixArtAlphaTextProjection, "forward", lambda self, x: torch.ones_like(text))
            assert torch.equal(m(t, None, pooled), times + 1)
        with monkeypatch.context() as p:
            p.setattr(QwenTimestepProjEmbeddings, "embed", staticmethod(lambda *a, **k: torch.ones_like(text)))
            assert torch.equal(m(t, None, pooled), 1 + text)
        with monkeypatch.context() as p:
            p.setitem(m.text_embedder.__dict__, "forward", lambda x: torch.ones_like(text))
            assert torch.equal(m(t, None, pooled), times + 1)
        assert torch.equal(m(t, None, pooled), times + text)
