"""Three projections of rows of their own in one launch of the tile kernel (odit_linear_three): against a float64 product, whole tiles and
tiles cut along the reduction (with and without scratch), tiles of all three problems at the ends of rows and features."""

import pytest
import torch

from vllm_omni_amd import _lib

pytestmark = pytest.mark.gpu

C = _lib.C
HANDWRITTEN = 2
# one rounding of the result, 2^-9 / sqrt(3) * (1.33 on average over a binade) in the 2-norm, and half as much again
_BOUND = {torch.bfloat16: 1.5 * 1.7e-3, torch.float16: 1.5 * 2.1e-4}


@pytest.mark.parametrize("rows, widths, K", [
    ((300, 257, 513), (264, 256, 8), 64),         # ragged rows and features, one step
    ((129, 8, 640), (1000, 520, 776), 320),       # the second problem less than a tile
    ((2706, 512, 512), (3072, 1024, 1024), 640),  # more than a round
    ((1024, 512, 256), (1024, 512, 512), 2048),   # cut along the reduction
])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("with_scratch", [True, False])
def test_three_projections(gpu, rows, widths, K, dtype, with_scratch):
    from vllm_omni_amd import kernels

    g = torch.Generator(device=gpu).manual_seed(sum(rows) + K)
    x = [torch.randn(m, K, device=gpu, generator=g).to(dtype) for m in rows]
    w = [(torch.randn(n, K, device=gpu, generator=g) * 0.05).to(dtype) for n in widths]
    b = [torch.randn(n, device=gpu, generator=g).to(dtype) for n in widths]
    out = [torch.full((m + 1, n), float("nan"), dtype=dtype, device=gpu) for m, n in zip(rows, widths)]
    q = (_lib.LinearProblem * 3)()
    for i in range(3):
        q[i].x, q[i].w, q[i].bias, q[i].out, q[i].M = x[i].data_ptr(), w[i].data_ptr(), b[i].data_ptr(), out[i].data_ptr(), rows[i]
        q[i].ldx = q[i].ldw = K
        q[i].ldo = widths[i]
    stream = torch.cuda.current_stream().cuda_stream
    ws = kernels._linear_scratch(gpu.index or 0, stream) if with_scratch else None
    print(f"three projections {dtype} rows={rows} widths={widths} K={K} scratch={with_scratch}", flush=True)

    def run(launch, flags=HANDWRITTEN, epilogue=(1, 1, 1)):
        return _lib.load().odit_linear_three(C.addressof(q), (C.c_int * 3)(*widths), K, (C.c_int * 3)(*epilogue), 0 if dtype == torch.bfloat16 else 1, flags,
                                             launch, ws.data_ptr() if ws is not None else None, ws.numel() if ws is not None else 0, stream)

    assert run(0) == 0
    assert all(bool(t.isnan().all()) for t in out), "asking launches nothing"
    assert run(1, flags=1) != 0, "the library has no such launch"
    assert run(1) == 0
    for i in range(3):
        y = x[i].double() @ w[i].double().t() + b[i].double()
        assert float((out[i][:-1].double() - y).norm() / y.norm()) < _BOUND[dtype]
        assert bool(out[i][-1].isnan().all()), "no row behind the last is written"
    if ws is not None:
        assert int(ws[:32768].view(torch.int32).abs().max().item()) == 0, "ticket words are handed back at zero"
