"""ODIT_LINEAR_FIRST: the library's first choice for a problem, until a tuning call has chosen a kernel."""

import pytest
import torch

from vllm_omni_amd import _lib, kernels

pytestmark = pytest.mark.gpu


def _first(x, w, b):
    lib, out = _lib.load(), torch.empty(x.shape[0], w.shape[0], dtype=x.dtype, device=x.device)
    ws = kernels._linear_workspace(lib, x.device)
    (M, K), N = x.shape, w.shape[0]
    _lib.check(lib.odit_linear_rows(x.data_ptr(), w.data_ptr(), b.data_ptr(), out.data_ptr(), None, None, M, N, K, K, K, N, 0,
                                    _lib.ODIT_EPI_BIAS, 0, 0, 0, 0, 4 | _lib.ODIT_LINEAR_LIBRARY, ws.data_ptr(), ws.numel(),
                                    torch.cuda.current_stream().cuda_stream), "odit_linear_rows")
    return out


# long reductions, which the library's kernels divide in different ways: other kernels give other bits
@pytest.mark.parametrize("M,N,K", [(2048, 3072, 12288), (3072, 2048, 8192)])
def test_first_choice_gives_way_to_a_tuned_kernel(gpu, M, N, K):
    g = torch.Generator(device=gpu).manual_seed(0)
    x, w, b = (torch.randn(s, device=gpu, generator=g).bfloat16() for s in ((M, K), (N, K), (N,)))
    kernels.linear(x, w, b, tune_iters=3, engine="library")
    tuned = kernels.linear(x, w, b, engine="library")
    assert torch.equal(_first(x, w, b), tuned)
