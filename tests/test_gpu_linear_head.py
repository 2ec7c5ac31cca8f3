"""A head's norm and projection in one launch (odit_linear_norm, 1024 to 3072 channels): against float64, at the ends of its tiles of rows and features and of the
batch entries, in each of its three tile widths."""

import pytest
import torch

import vllm_omni_amd.blocks.qwen_image  # noqa: F401  (names the module classes that native calls take)
from vllm_omni_amd import kernels

pytestmark = pytest.mark.gpu

# Two roundings, of the normed rows and of the result, each 2^-9 / sqrt(3) * (1.33 on average over a binade) in the 2-norm, and half as much again
_BOUND = {torch.bfloat16: 1.5 * 2.0 ** 0.5 * 1.7e-3, torch.float16: 1.5 * 2.0 ** 0.5 * 2.1e-4}


@pytest.mark.parametrize("B, S, C, N, bias", [
    (1, 1, 3072, 64, True), (2, 15, 3072, 64, True), (3, 17, 1024, 8, False), (1, 1025, 3072, 24, True),  # 16 features to a tile
    (2, 700, 3072, 64, True), (1, 2047, 2048, 40, False),  # 32
    (1, 4096, 3072, 64, True), (2, 4095, 3072, 64, False), (3, 1700, 1024, 64, True),  # 64, one round and two
])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_head(gpu, B, S, C, N, bias, dtype):
    print(f"head {B}x{S}x{C} N={N} bias={bias} {dtype}", flush=True)
    g = torch.Generator(device=gpu).manual_seed(S)
    lin = torch.nn.Linear(C, N, bias=bias, device=gpu, dtype=dtype).requires_grad_(False)
    with torch.no_grad():
        for p in lin.parameters():
            p.normal_(0.0, 0.05, generator=g)
    x = (torch.randn(B, S, C, device=gpu, generator=g) + 3 * torch.randn(B, S, 1, device=gpu, generator=g)).to(dtype)  # (rows with a mean)
    scale, shift = torch.randn(B, 2 * C, device=gpu, generator=g).to(dtype).chunk(2, dim=1)
    with torch.inference_mode():
        got = kernels.project_normed(lin, x, shift, scale, 1e-6)
        assert got is not None
        apart = kernels.project(lin, kernels.adaln_modulate(x, shift, scale, eps=1e-6))
        exact = torch.nn.functional.layer_norm(x.double(), (C,), eps=1e-6) * (1 + scale.double()[:, None]) + shift.double()[:, None]
        exact = torch.nn.functional.linear(exact, lin.weight.double(), lin.bias.double() if bias else None)
    # Every batch entry and the last rows by themselves; the 2-norm of n roundings scatters by 1 / sqrt(2 n) or a little more of itself: six times 1 / sqrt(n)
    for rows in (got, apart):
        for b in range(B):
            assert float((rows[b].double() - exact[b]).norm() / exact[b].norm()) < _BOUND[dtype] * (1 + (S * N) ** -0.5 * 6)
        assert float((rows[:, -1].double() - exact[:, -1]).norm() / exact[:, -1].norm()) < _BOUND[dtype] * (1 + (B * N) ** -0.5 * 6)


def test_refused(gpu):
    def call(C, N, M):
        lin = torch.nn.Linear(C, N, device=gpu, dtype=torch.bfloat16).requires_grad_(False)
        x, head = torch.ones(1, M, C, device=gpu, dtype=torch.bfloat16), torch.ones(1, 2 * C, device=gpu, dtype=torch.bfloat16)
        with torch.inference_mode():
            return kernels.project_normed(lin, x, head[:, :C], head[:, C:], 1e-6)

    assert call(3072, 64, 64) is not None
    assert call(3072, 72, 64) is None and call(1536, 64, 64) is None and call(4096, 64, 64) is None  # features and widths that it has no tile for
    assert call(3072, 64, 16384) is None  # more than two rounds


@pytest.mark.parametrize("C, N", [(3072, 72), (1536, 64), (4096, 64), (320, 64)])
def test_refused_widths_cost_no_memory(gpu, C, N):
    lin = torch.nn.Linear(C, N, device=gpu, dtype=torch.bfloat16).requires_grad_(False)
    x, head = torch.ones(1, 64, C, device=gpu, dtype=torch.bfloat16), torch.ones(1, 2 * C, device=gpu, dtype=torch.bfloat16)
    with torch.inference_mode():
        assert kernels.project_normed(lin, x, head[:, :C], head[:, C:], 1e-6) is None
        torch.cuda.reset_peak_memory_stats()
        before = torch.cuda.memory_allocated()
        assert kernels.project_normed(lin, x, head[:, :C], head[:, C:], 1e-6) is None
        assert torch.cuda.max_memory_allocated() == before
