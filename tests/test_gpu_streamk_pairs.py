"""Two problems in one launch of the stream-K kernel (csrc/gemm_bf16.hip): the form that runs is the one whose time the choice of a kernel goes by, which counts in what a
pair's shared tiles cost; each width of tile, alone on its tiles and sharing them, against float64."""

import pytest
import torch

from vllm_omni_amd import _lib, kernels

pytestmark = pytest.mark.gpu

# one rounding of the result, 2^-9 / sqrt(3) * (1.33 on average over a binade) in the 2-norm, and half as much again
_BOUND = {torch.bfloat16: 1.5 * 1.7e-3, torch.float16: 1.5 * 2.1e-4}


# Times (us) by the plan at 256 CUs, 128 / 192 / 256 wide, shared by whole workgroups or in ranges that run on; one problem's times would choose the width noted last
@pytest.mark.parametrize("rows, N, K, width", [
    ((195, 256), 3072, 3072, 128),   # 24.1 / 31.9 / 31.9; 192
    ((128, 40), 9216, 3072, 128),    # 30.7 / 30.8 / 36.3; 256
    ((300, 300), 3072, 3072, 192),   # 31.4 / 30.8 / 36.3; 256
    ((256, 64), 9216, 3072, 256),    # 37.8 / 38.7 / 37.1; 256
    ((512, 80), 9216, 3072, 192),    # 56.2 / 43.5 / 50.2; 192
    ((1, 129), 136, 128, 128),       # two steps
])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_form_and_results(gpu, rows, N, K, width, dtype):
    print(f"pair {rows} N={N} K={K} {dtype}", flush=True)
    g = torch.Generator(device=gpu).manual_seed(K)
    q, ops = (_lib.LinearProblem * 2)(), []
    for i, M in enumerate(rows):
        x, w, b = torch.randn(M, K, device=gpu, generator=g).to(dtype), (torch.randn(N, K, device=gpu, generator=g) * 0.05).to(dtype), torch.randn(N, device=gpu, generator=g).to(dtype)
        ops.append((x, w, b, torch.full((M + 1, N), float("nan"), dtype=dtype, device=gpu)))
        q[i].x, q[i].w, q[i].bias, q[i].out, q[i].M = (*(t.data_ptr() for t in ops[i]), M)
        q[i].ldx = q[i].ldw = K
        q[i].ldo = N
    stream = torch.cuda.current_stream().cuda_stream
    ws = kernels._linear_scratch(gpu.index or 0, stream)

    def run():
        _lib.check(_lib.load().odit_linear_pair(_lib.C.addressof(q), N, K, _lib.ODIT_EPI_BIAS, 0, 0 if dtype == torch.bfloat16 else 1, _lib.ODIT_LINEAR_HANDWRITTEN,
                                                ws.data_ptr(), ws.numel(), stream), "odit_linear_pair")
        torch.cuda.synchronize()

    run()
    for x, w, b, out in ops:
        y = x.double() @ w.double().t() + b.double()
        assert float((out[:-1].double() - y).norm() / y.norm()) < _BOUND[dtype] * (1 + (len(y) * N) ** -0.5 * 6)
        assert bool(out[-1].isnan().all())
    if torch.cuda.get_device_properties(gpu).multi_processor_count == 256:
        with torch.profiler.profile(activities=[torch.profiler.ProfilerActivity.CUDA]) as p:
            run()
        names = [e.name for e in p.events() if "gemm" in e.name]
        assert len(names) == 1 and "gemm_streamk_kernel" in names[0] and f", 128, {width}>" in names[0], names
