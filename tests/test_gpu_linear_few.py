"""Projections of a few rows (``odit_linear_few``) against float32 on the GPU."""

import pytest
import torch
import torch.nn.functional as F

from vllm_omni_amd import kernels

pytestmark = pytest.mark.gpu


# reduction shares of 0, 1, part of and several groups of loads per wave; features that end inside a tile; more tiles than
# workgroups; one, the most and too many rows
@pytest.mark.parametrize("N,K", [(16, 32), (77, 64), (256, 256), (3072, 320), (6144, 3072), (129, 5120), (20000, 288)])
@pytest.mark.parametrize("M", [1, 2, 5, 16, 17])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_linear_few(M, N, K, dtype):
    g = torch.Generator(device="cuda").manual_seed(M * N + K)
    x = torch.randn(M, K, device="cuda", generator=g).to(dtype)
    w = (torch.randn(N, K + 8, device="cuda", generator=g) * K ** -0.5).to(dtype)[:, :K]
    b = torch.randn(N, device="cuda", generator=g).to(dtype)
    tol = 6e-3 if dtype == torch.bfloat16 else 8e-4
    for bias in (b, None):
        for silu in (False, True):
            a = kernels.silu(x) if silu else x
            ref = F.linear(a.float(), w.float(), None if bias is None else bias.float())
            out = kernels.linear_few(x, w, bias, silu_input=silu)
            assert out.dtype == dtype and out.shape == (M, N)
            torch.testing.assert_close(out.float(), ref, rtol=tol, atol=tol)


# up to 4 rows and K a multiple of 512: rows of W two or four at a time (four from 65536 on), with a remainder and with fewer
# than a wavefront, a workgroup or the grid takes; one chunk of 512, an odd number of them
@pytest.mark.parametrize("N,K", [(1, 512), (2, 1024), (15, 512), (17, 3584), (12289, 1536), (65535, 512), (65539, 1024), (147459, 512)])
@pytest.mark.parametrize("M", [1, 2, 3, 4, 5])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_linear_few_by_whole_rows(M, N, K, dtype):
    g = torch.Generator(device="cuda").manual_seed(M * N + K)
    x = torch.randn(M, K + 8, device="cuda", generator=g).to(dtype)[:, :K]
    w = (torch.randn(N, K + 16, device="cuda", generator=g) * K ** -0.5).to(dtype)[:, :K]
    w[N // 2, K - 1] = float("inf")
    b = torch.randn(N, device="cuda", generator=g).to(dtype)
    a = kernels.silu(x.contiguous())
    want = a.double() @ w.double().t() + b.double()
    out = kernels.linear_few(x, w, b, silu_input=True).double()
    assert torch.equal(out[:, N // 2], want[:, N // 2])  # an infinity of the sign of x, and of that feature only
    keep = torch.arange(N, device="cuda") != N // 2
    # one rounding of a float32 sum: half a step of the type, relative; the sum's own error is below 1e-5 of |x| |w|
    tol = 2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -11
    torch.testing.assert_close(out[:, keep], want[:, keep], rtol=tol, atol=2e-5)
    assert torch.equal(out, kernels.linear_few(x, w, b, silu_input=True).double())
