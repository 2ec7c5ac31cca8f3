"""The tile kernel at the ends of its operands: rows and features of padding in dense and strided operands, in one tensor and two, change no row of the result, and
none behind the last is written, whatever lies behind the operand. (Where they are fetched from: test_tile_plans.py.)"""

import pytest
import torch

from vllm_omni_amd import _lib

pytestmark = pytest.mark.gpu

HANDWRITTEN = 2
# one rounding of the result, 2^-9 / sqrt(3) * (1.33 on average over a binade) in the 2-norm, and half as much again
_BOUND = {torch.bfloat16: 1.5 * 1.7e-3, torch.float16: 1.5 * 2.1e-4}


def _rows(gpu, rows, K, pad, dtype, scale, seed):
    """[rows, K] of row stride K + pad, NaN in the gaps and behind the last row."""
    g = torch.Generator(device=gpu).manual_seed(seed)
    t = torch.full((rows + 300, K + pad), float("nan"), dtype=dtype, device=gpu)
    t[:rows, :K] = (torch.randn(rows, K, device=gpu, generator=g) * scale).to(dtype)
    return t[:rows, :K]


@pytest.mark.parametrize("M, N, K", [(1025, 3072, 64), (1279, 264, 640), (2706, 5128, 320), (8193, 520, 64), (4000, 3080, 1024)])
@pytest.mark.parametrize("pad", [0, 24])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_rows_of_padding(gpu, M, N, K, pad, dtype):
    from vllm_omni_amd import kernels

    x, w = _rows(gpu, M, K, pad, dtype, 1, M), _rows(gpu, N, K, pad, dtype, 0.05, N)
    out = torch.full((M + 1, N), float("nan"), dtype=dtype, device=gpu)
    stream = torch.cuda.current_stream().cuda_stream
    ws = kernels._linear_scratch(gpu.index or 0, stream)
    print(f"padding {dtype} M={M} N={N} K={K} pad={pad}", flush=True)
    _lib.check(_lib.load().odit_linear_rows(x.data_ptr(), w.data_ptr(), None, out.data_ptr(), None, None, M, N, K, K + pad, K + pad, N, 0, _lib.ODIT_EPI_NONE, 2,
                                            0 if dtype == torch.bfloat16 else 1, 0, 0, HANDWRITTEN, ws.data_ptr(), ws.numel(), stream), "odit_linear_rows")
    y = x.double() @ w.double().t()
    assert float((out[:-1].double() - y).norm() / y.norm()) < _BOUND[dtype]
    assert bool(out[-1].isnan().all()), "no row behind the last is written"


@pytest.mark.parametrize("M", [1536, 1500, 2305])
def test_rows_of_padding_in_two_tensors(gpu, M):
    from vllm_omni_amd import kernels

    N, K, K2 = 3072, 3072, 3072
    x, x2, w = _rows(gpu, M, K, 8, torch.bfloat16, 1, 1), _rows(gpu, M, K2, 0, torch.bfloat16, 1, 2), _rows(gpu, N, K + K2, 0, torch.bfloat16, 0.05, 3)
    residual = _rows(gpu, M, N, 0, torch.bfloat16, 1, 4)
    out = torch.full((M + 1, N), float("nan"), dtype=torch.bfloat16, device=gpu)
    stream = torch.cuda.current_stream().cuda_stream
    ws = kernels._linear_scratch(gpu.index or 0, stream)
    print(f"padding in two tensors M={M}", flush=True)
    _lib.check(_lib.load().odit_linear_join(x.data_ptr(), x2.data_ptr(), w.data_ptr(), None, out.data_ptr(), residual.data_ptr(), None, M, N, K, K2, K + 8, K2, K + K2,
                                            N, N, _lib.ODIT_EPI_GATED_RESIDUAL, 0, 0, 0, 0, 0, ws.data_ptr(), ws.numel(), stream), "odit_linear_join")
    y = torch.cat([x, x2], 1).double() @ w.double().t() + residual.double()
    assert float((out[:-1].double() - y).norm() / y.norm()) < _BOUND[torch.bfloat16]
    assert bool(out[-1].isnan().all())
