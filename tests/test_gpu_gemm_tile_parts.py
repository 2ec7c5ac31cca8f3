"""Tiles of 128 rows cut into more parts than they have quadrants (csrc/gemm_tile.h, 5 to 8), of which the later ones finish none: against a float64 product,
run after run the same bits, ticket words handed back, heads at a cut tile's end."""

import pytest
import torch

from vllm_omni_amd import _lib
from test_gpu_linear_heads import _check, _Problem, _run

pytestmark = pytest.mark.gpu

# one rounding of the result, 2^-9 / sqrt(3) * (1.33 on average over a binade) in the 2-norm, and half as much again
_BOUND = {torch.bfloat16: 1.5 * 1.7e-3, torch.float16: 1.5 * 2.1e-4}


@pytest.fixture()
def scratch(gpu):
    from vllm_omni_amd import kernels

    ws = kernels._linear_scratch(gpu.index or 0, torch.cuda.current_stream().cuda_stream)
    yield ws
    assert int(ws[:32768].view(torch.int32).abs().max().item()) == 0, "ticket words are handed back at zero"


# (rows, features, reduction, parts; test_tile_plans.py holds the plan to them)
PARTS = [
    (1100, 1280, 12288, 5),  # 45 tiles
    (1700, 704, 12288, 6),   # 42
    (1100, 1000, 12352, 7),  # 36, parts of 27 and 28 steps
    (1025, 520, 8192, 8),    # 27, one row in the last tile
    (1100, 8, 1408, 6),      # 9, parts of 3 and 4 steps
]
HEADS = [(300, 100, 3, 8192, 8), (500, 9, 4, 8192, 8), (640, 9, 4, 8192, 7)]  # (rows of two, heads of 128, reduction, parts)


@pytest.mark.parametrize("M, N, K, parts", PARTS)
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_parts(scratch, gpu, M, N, K, parts, dtype):
    from vllm_omni_amd import kernels

    print(f"{parts} parts {dtype} {M}x{N}x{K}", flush=True)
    g = torch.Generator(device=gpu).manual_seed(N)
    x, w, b = torch.randn(M, K, device=gpu, generator=g).to(dtype), (torch.randn(N, K, device=gpu, generator=g) * 0.05).to(dtype), torch.randn(N, device=gpu, generator=g).to(dtype)
    residual = torch.randn(M, N, device=gpu, generator=g).to(dtype)
    y = x.double() @ w.double().t() + b.double()
    got, added = (kernels.linear(x, w, b, residual=r, engine="handwritten") for r in (None, residual))
    assert float((got.double() - y).norm() / y.norm()) < _BOUND[dtype]
    y += residual.double()
    assert float((added.double() - y).norm() / y.norm()) < _BOUND[dtype]
    for _ in range(20):  # (whoever arrives last, and whoever gives up)
        assert torch.equal(added, kernels.linear(x, w, b, residual=residual, engine="handwritten"))


@pytest.mark.parametrize("S0, S1, H, K, parts", HEADS)
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_heads(scratch, gpu, S0, S1, H, K, parts, dtype):
    print(f"heads of {parts} parts {dtype} {S0}+{S1} rows, {H} heads, K={K}", flush=True)
    ps = [_Problem(gpu, dtype, 1, S0, K, H, 128, seed=1), _Problem(gpu, dtype, 1, S1, K, H, 128, seed=2)]
    joint = [torch.full((1, S0 + S1, H, 128), float("nan"), dtype=dtype, device=gpu) for _ in range(3)]
    for _ in range(2):
        _lib.check(_run(ps, (S1, 0), joint, K, dtype, scratch, flags=_lib.ODIT_LINEAR_HANDWRITTEN), "odit_linear_heads")
        _check(ps, (S1, 0), joint, dtype)
