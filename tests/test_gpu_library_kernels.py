"""Which of the library's kernels run: never its hand-scheduled one ("Custom_..."), which now and then gives other results for the same operands and is its own first
choice for all of these problems; and what runs in its place."""

import pytest
import torch

from vllm_omni_amd import _lib, kernels

pytestmark = pytest.mark.gpu

LIBRARY, FIRST, NO_TILE = _lib.ODIT_LINEAR_LIBRARY, 4, _lib.ODIT_LINEAR_NO_TILE
BIAS, GELU, GATED, RESIDUAL = _lib.ODIT_EPI_BIAS, _lib.ODIT_EPI_BIAS_GELU_TANH, _lib.ODIT_EPI_GATED_RESIDUAL_PRE, _lib.ODIT_EPI_GATED_RESIDUAL
# one rounding of the result, 2^-9 / sqrt(3) * (1.33 on average over a binade) in the 2-norm, and half as much again
_BOUND = {torch.bfloat16: 1.5 * 1.7e-3, torch.float16: 1.5 * 2.1e-4}


class _Problem:
    def __init__(self, gpu, M, N, K, epilogue, dtype, groups=1):
        g = torch.Generator(device=gpu).manual_seed(M + N + K)
        self.M, self.N, self.K, self.epilogue, self.dtype, self.groups = M, N, K, epilogue, dtype, groups
        self.x, self.w = torch.randn(M, K, device=gpu, generator=g).to(dtype), (torch.randn(N, K, device=gpu, generator=g) * 0.02).to(dtype)
        self.gate = torch.randn(groups, N, device=gpu, generator=g)
        self.bias = torch.randn(N, device=gpu, generator=g).to(dtype)
        self.gate_bias = self.gate * self.bias.float()
        self.residual = torch.randn(M, N, device=gpu, generator=g).to(dtype)

    def run(self, flags):
        gated, added = self.epilogue == GATED, self.epilogue in (GATED, RESIDUAL)
        out = torch.empty(self.M, self.N, dtype=self.dtype, device=self.x.device)
        stream = torch.cuda.current_stream().cuda_stream
        ws = kernels._linear_scratch(self.x.device.index or 0, stream)
        _lib.check(_lib.load().odit_linear_rows(
            self.x.data_ptr(), self.w.data_ptr(), (self.gate_bias if gated else self.bias).data_ptr(), out.data_ptr(), self.residual.data_ptr() if added else None,
            self.gate.data_ptr() if gated else None, self.M, self.N, self.K, self.K, self.K, self.N, self.N, self.epilogue, 2, 0 if self.dtype == torch.bfloat16 else 1,
            self.M // self.groups if gated and self.groups > 1 else 0, self.N, flags, ws.data_ptr(), ws.numel(), stream), "odit_linear_rows")
        return out

    def names(self, flags):
        self.run(flags)
        torch.cuda.synchronize()
        with torch.profiler.profile(activities=[torch.profiler.ProfilerActivity.CUDA]) as p:
            out = self.run(flags)
            torch.cuda.synchronize()
        return out, [e.name for e in p.events() if "gemm" in e.name or "Cijk" in e.name]

    def exact(self):
        y = self.x.double() @ self.w.double().t() + self.bias.double()
        if self.epilogue == GELU:
            return torch.nn.functional.gelu(y, approximate="tanh")
        return y if self.epilogue == BIAS else self.residual.double() + (y.view(self.groups, -1, self.N) * self.gate.double()[:, None]).flatten(0, 1)


@pytest.mark.parametrize("M, N, K, epilogue, groups", [
    (2048, 15360, 5120, BIAS, 1),    # it would sum every tile whole
    (8192, 9216, 3072, BIAS, 1),     # it would split tiles
    (4608, 12288, 3072, GELU, 1),
    (16384, 5120, 5120, GATED, 2),   # a launch for each group of rows
])
@pytest.mark.parametrize("flags", [0, FIRST, NO_TILE, LIBRARY, LIBRARY | FIRST])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_hand_scheduled_kernel_never_runs(gpu, M, N, K, epilogue, groups, flags, dtype):
    print(f"library kernels {dtype} {M}x{N}x{K} epilogue={epilogue} flags={flags}", flush=True)
    p = _Problem(gpu, M, N, K, epilogue, dtype, groups)
    out, names = p.names(flags)
    assert names and not any(n.startswith("Custom") for n in names), names
    y = p.exact()
    assert float((out.double() - y).norm() / y.norm()) < _BOUND[dtype]


@pytest.mark.parametrize("M", [2048, 7072])
def test_in_its_place_the_tile_kernel_with_the_library_s_bits(gpu, M):
    """A call that keeps the library's order of summation: the tile kernel, with the bits of the library's kernels that split no tile."""
    p = _Problem(gpu, M, 15360, 5120, BIAS, torch.bfloat16)
    out, names = p.names(FIRST)
    assert len(names) == 1 and "gemm_tile_kernel" in names[0], names
    assert torch.equal(out, p.run(LIBRARY | FIRST))


@pytest.mark.parametrize("M, N", [(3261, 13824), (7072, 13824), (2875, 15360)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_gelu_in_its_place(gpu, M, N, dtype):
    """The sums of whole tiles, and GELU as the library computes it: x = a power of two times one row of W, so that it is exact."""
    p = _Problem(gpu, M, N, 5120, GELU, dtype)
    out, names = p.names(FIRST)
    assert len(names) == 1 and "gemm_tile_kernel" in names[0], names
    assert len(p.names(LIBRARY | FIRST)[1]) == 1
    p.x.zero_()
    p.x[torch.arange(M, device=gpu), torch.randint(0, 5120, (M,), device=gpu)] = 64.0
    assert torch.equal(p.run(FIRST), p.run(LIBRARY | FIRST))  # (the library's next kernel may sum in another order, but one term is one term)


@pytest.mark.parametrize("M", [3261, 4800])  # (whole tiles; some of them parted)
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_gelu_of_extremes(gpu, M, dtype):
    p = _Problem(gpu, M, 13824, 5120, GELU, dtype)
    top = torch.finfo(dtype).max
    values = [-float("inf"), float("inf"), float("nan"), -top, top / 4, -100.0, -20.0, -9.0, -6.0, -0.0, 0.0, torch.finfo(dtype).tiny, -torch.finfo(dtype).tiny]
    p.x.zero_()
    p.bias.zero_()
    p.bias[:len(values) + 1] = torch.tensor(values + [top], dtype=dtype, device=gpu)
    own, library = p.run(FIRST), p.run(LIBRARY | FIRST)
    n = len(values)
    assert torch.equal(own[:, n], torch.full_like(own[:, n], top))  # (the library's bf16 overflows there)
    own[:, n] = library[:, n] = 0
    assert torch.equal(own.isnan(), library.isnan())
    assert torch.equal(torch.where(own.isnan(), 0, own.view(torch.int16)), torch.where(library.isnan(), 0, library.view(torch.int16)))


@pytest.mark.parametrize("epilogue", [GATED, RESIDUAL])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_gated_and_residual_epilogues_with_the_library_s_bits(gpu, epilogue, dtype):
    """Two entries of a batch whose gates change inside a tile, 10 rounds of whole tiles."""
    p = _Problem(gpu, 32760, 5120, 5120, epilogue, dtype, 2)
    out, names = p.names(FIRST)
    assert len(names) == 1 and "gemm_tile_kernel" in names[0], names
    assert torch.equal(out, p.run(LIBRARY | FIRST))
    own = p.run(0)  # (who names nothing keeps the tile kernel's own order of operations)
    assert 0 < float((own != out).double().mean()) < 1e-3


def test_a_tuning_call_does_not_choose_it(gpu):
    p = _Problem(gpu, 1280, 5120, 1024, BIAS, torch.bfloat16)
    kernels.linear(p.x, p.w, p.bias, tune_iters=2, engine="library")
    _, names = p.names(LIBRARY)
    assert names and not any(n.startswith("Custom") for n in names), names


@pytest.mark.parametrize("B", [1, 2])
def test_image_conditioned_video(gpu, B):
    """A block that runs operation by operation (its cross-attention has image tokens too)."""
    from vllm_omni_amd.blocks.wan import WanTransformerBlock

    g = torch.Generator(device=gpu).manual_seed(B)
    with torch.device(gpu):
        block = WanTransformerBlock(5120, 13824, 40, added_kv_proj_dim=5120, cross_attn_norm=True).bfloat16().eval()
    with torch.no_grad():
        for p in block.parameters():
            p.normal_(0.0, 0.02, generator=g)
    x, ctx = torch.randn(B, 7072 // B, 5120, device=gpu, generator=g).bfloat16(), torch.randn(B, 257 + 512, 5120, device=gpu, generator=g).bfloat16()
    temb = torch.randn(B, 6, 5120, device=gpu, generator=g).bfloat16()
    with torch.inference_mode():
        out = block(x, ctx, temb)
        torch.cuda.synchronize()
        with torch.profiler.profile(activities=[torch.profiler.ProfilerActivity.CUDA]) as p:
            again = block(x, ctx, temb)
            torch.cuda.synchronize()
    names = [e.name for e in p.events()]
    assert names and not any(n.startswith("Custom") for n in names), names
    assert torch.equal(out, again)
