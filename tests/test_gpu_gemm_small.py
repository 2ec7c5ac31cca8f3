"""The kernel for small products (csrc/gemm_small.hip) at the edges of its tiles and of its stages, one problem and two, against a
float64 product. The bound is the one of test_gpu_gemm_tile.py: 1.5 times the rounding of the result."""

import pytest
import torch

pytestmark = pytest.mark.gpu

_BOUND = {torch.bfloat16: 2.5e-3, torch.float16: 3.2e-4}


def _rel(got, want):
    assert torch.isfinite(got).all()
    return ((got.double() - want).norm() / want.norm()).item()


def _mk(gpu, M, N, K, dtype, seed):
    g = torch.Generator(device=gpu).manual_seed(seed)
    x = torch.randn(M, K, device=gpu, generator=g).to(dtype)
    w = (torch.randn(N, K, device=gpu, generator=g) * 0.05).to(dtype)
    b = torch.randn(N, device=gpu, generator=g).to(dtype)
    return x, w, b, x.double() @ w.double().t()


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("M0,M1,N,K", [
    (1, 1, 256, 64),       # one step, one row
    (65, 63, 264, 128),    # one row over, ragged features, two steps
    (256, 64, 768, 256),   # four steps
    (300, 129, 200, 320),  # five: eight stages, all in flight
    (256, 64, 256, 512),   # eight
    (256, 64, 256, 576),   # nine: the first stage is filled again
    (200, 33, 328, 2048),  # the longest
    (1984, 64, 1024, 256), # two workgroups to a CU
])
def test_small_gemm(gpu, dtype, M0, M1, N, K):
    """Two problems in one launch, then each alone: the same bits."""
    from vllm_omni_amd import _lib, kernels

    lib, code = _lib.load(), 0 if dtype == torch.bfloat16 else 1
    ws = kernels._linear_scratch(gpu.index or 0, torch.cuda.current_stream().cuda_stream)
    ops = [_mk(gpu, m, N, K, dtype, m + i) for i, m in enumerate((M0, M1))]
    g = torch.Generator(device=gpu).manual_seed(9)
    res = [torch.randn(m, N, device=gpu, generator=g).to(dtype) for m in (M0, M1)]
    rows = [max(1, m // 2) for m in (M0, M1)]
    gates = [torch.randn(-(-m // r), N, device=gpu, generator=g) for m, r in zip((M0, M1), rows)]
    scaled = [t * o[2].float() for t, o in zip(gates, ops)]
    out = [torch.full((m, N), float("nan"), dtype=dtype, device=gpu) for m in (M0, M1)]

    def run(epilogue, flags=0):
        q = (_lib.LinearProblem * 2)()
        for i, m in enumerate((M0, M1)):
            q[i].x, q[i].w, q[i].bias, q[i].out, q[i].M = ops[i][0].data_ptr(), ops[i][1].data_ptr(), ops[i][2].data_ptr(), out[i].data_ptr(), m
            q[i].ldx, q[i].ldw, q[i].ldo, q[i].ldr = K, K, N, N
            if epilogue == 5:
                q[i].bias, q[i].residual, q[i].gate = scaled[i].data_ptr(), res[i].data_ptr(), gates[i].data_ptr()
                q[i].rows_per_gate, q[i].gate_stride = rows[i], N
        rc = lib.odit_linear_pair(_lib.C.addressof(q), N, K, epilogue, 2, code, flags, ws.data_ptr(), ws.numel(), torch.cuda.current_stream().cuda_stream)
        _lib.check(rc, "odit_linear_pair")
        return [t.clone() for t in out]

    plain = [o[3] + o[2].double() for o in ops]
    got = run(1)
    assert all(_rel(a, b) < _BOUND[dtype] for a, b in zip(got, plain))
    if K <= 1024:
        for (x, w, b, _), a in zip(ops, got):
            assert torch.equal(a, kernels.linear(x, w, b))
    gelu = run(3)
    assert all(_rel(a, torch.nn.functional.gelu(b, approximate="tanh")) < _BOUND[dtype] for a, b in zip(gelu, plain))
    per_row = [t[torch.arange(m, device=gpu) // r].double() for t, m, r in zip(gates, (M0, M1), rows)]
    want = [r.double() + p * y for r, p, y in zip(res, per_row, plain)]
    assert all(_rel(a, b) < _BOUND[dtype] for a, b in zip(run(5), want))
