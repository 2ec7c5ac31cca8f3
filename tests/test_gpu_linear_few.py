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
