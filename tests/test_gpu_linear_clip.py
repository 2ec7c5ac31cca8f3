"""ODIT_LINEAR_CLIP: the gated epilogues of float16 clip what they write. The bits of the same call without the flag and a clip behind it, by every
kernel that such a projection has, for one problem, two and one over two tensors."""

import pytest
import torch

from vllm_omni_amd import _lib

pytestmark = pytest.mark.gpu

C = _lib.C
LIBRARY, HANDWRITTEN, CLIP, CLIP2 = _lib.ODIT_LINEAR_LIBRARY, _lib.ODIT_LINEAR_HANDWRITTEN, _lib.ODIT_LINEAR_CLIP, _lib.ODIT_LINEAR_CLIP2
PRE = _lib.ODIT_EPI_GATED_RESIDUAL_PRE


def _operands(gpu, M, N, K, pad=0):
    g = torch.Generator(device=gpu).manual_seed(M + N + K)
    x = torch.randn(M, K, device=gpu, generator=g).half()
    w = (torch.randn(N, K, device=gpu, generator=g) * 0.05).half()
    residual = (torch.randn(M, N, device=gpu, generator=g).sign() * 65500).half()  # half of the results are past the largest finite value
    residual[:, ::3] = torch.randn(M, (N + 2) // 3, device=gpu, generator=g).half()
    residual[M // 2, N // 2] = float("nan")
    residual[M - 1, N - 1], residual[0, 0] = float("inf"), float("-inf")
    gate, bias = 20 * torch.randn(N, device=gpu, generator=g), torch.randn(N, device=gpu, generator=g)
    return x, w, residual, gate, bias, torch.zeros(M, N + pad, dtype=torch.half, device=gpu)


def _same(got, plain):
    want = plain.clamp(-65504, 65504)
    assert bool(torch.isinf(plain).any()) and bool(plain.isnan().any())
    assert torch.equal(got.isnan(), want.isnan()) and torch.equal(got.nan_to_num(7.0), want.nan_to_num(7.0))


@pytest.mark.parametrize("M, N, K, flags", [
    (300, 264, 256, LIBRARY), (33, 260, 64, LIBRARY),  # (rows that the clip takes whole, and rows that it cannot)
    (100, 512, 256, HANDWRITTEN), (513, 264, 1024, HANDWRITTEN),       # stream-K
    (1281, 264, 64, HANDWRITTEN), (1100, 3072, 3072, HANDWRITTEN),     # the tile kernel, whole tiles and cut ones
    (65, 72, 256, 0), (257, 1024, 1024, 0),                             # as the call chooses: the small kernel
])
@pytest.mark.parametrize("pad", [0, 12])
def test_one_projection(gpu, M, N, K, flags, pad):
    from vllm_omni_amd import kernels

    x, w, residual, gate, bias, out = _operands(gpu, M, N, K, pad if flags == LIBRARY else 2 * pad // 3)
    stream = torch.cuda.current_stream().cuda_stream
    ws = kernels._linear_scratch(gpu.index or 0, stream)
    print(f"clip M={M} N={N} K={K} flags={flags} pad={pad}", flush=True)

    def run(flags):
        out.zero_()
        _lib.check(_lib.load().odit_linear_rows(x.data_ptr(), w.data_ptr(), bias.data_ptr(), out.data_ptr(), residual.data_ptr(), gate.data_ptr(), M, N, K, K, K,
                                                out.stride(0), N, PRE, 2, 1, 0, 0, flags, ws.data_ptr(), ws.numel(), stream), "odit_linear_rows")
        return out.clone()

    plain, got = run(flags), run(flags | CLIP)
    _same(got[:, :N], plain[:, :N])
    assert not bool(got[:, N:].any())


@pytest.mark.parametrize("rows, N, K", [((512, 80), 3072, 3072), ((130, 65), 256, 256), ((810, 466), 3072, 3072)])
@pytest.mark.parametrize("flags", [CLIP, CLIP2, CLIP | CLIP2])
def test_two_projections(gpu, rows, N, K, flags):
    from vllm_omni_amd import kernels

    ops = [_operands(gpu, m, N, K) for m in rows]
    q = (_lib.LinearProblem * 2)()
    for i, (x, w, residual, gate, bias, out) in enumerate(ops):
        q[i].x, q[i].w, q[i].bias, q[i].residual, q[i].gate, q[i].out, q[i].M = (*(t.data_ptr() for t in (x, w, bias, residual, gate, out)), rows[i])
        q[i].ldx = q[i].ldw = K
        q[i].ldo = q[i].ldr = N
    stream = torch.cuda.current_stream().cuda_stream
    ws = kernels._linear_scratch(gpu.index or 0, stream)
    print(f"clip rows={rows} N={N} K={K} flags={flags}", flush=True)

    def run(flags):
        _lib.check(_lib.load().odit_linear_pair(C.addressof(q), N, K, PRE, 2, 1, flags, ws.data_ptr(), ws.numel(), stream), "odit_linear_pair")
        return [o[-1].clone() for o in ops]

    plain, got = run(0), run(flags)
    for i, bit in enumerate((CLIP, CLIP2)):
        if flags & bit:
            _same(got[i], plain[i])
        else:
            assert torch.equal(got[i].nan_to_num(7.0, 9.0, -9.0), plain[i].nan_to_num(7.0, 9.0, -9.0)), "the other problem's rows are as they come"


@pytest.mark.parametrize("M", [1536, 1500])
def test_two_tensors(gpu, M):
    from vllm_omni_amd import kernels

    N, K, K2 = 3072, 3072, 3072
    x, w, residual, gate, bias, out = _operands(gpu, M, N, K + K2)
    x2 = x[:, K:].contiguous()
    stream = torch.cuda.current_stream().cuda_stream
    ws = kernels._linear_scratch(gpu.index or 0, stream)

    def run(flags):
        _lib.check(_lib.load().odit_linear_join(x.data_ptr(), x2.data_ptr(), w.data_ptr(), bias.data_ptr(), out.data_ptr(), residual.data_ptr(), gate.data_ptr(), M, N, K,
                                                K2, K + K2, K2, K + K2, N, N, PRE, 2, 1, 0, 0, flags, ws.data_ptr(), ws.numel(), stream), "odit_linear_join")
        return out.clone()

    plain, got = run(0), run(CLIP)
    _same(got, plain)


# a gate vector for every group of rows: the library's launch for each (the last one shorter), the stream-K kernel, and the tile kernel's groups that change inside a tile and
# at its end, whole and cut
@pytest.mark.parametrize("M, rows, N, K, flags", [
    (300, 130, 264, 256, LIBRARY), (400, 200, 1024, 512, LIBRARY), (33, 7, 260, 64, LIBRARY),
    (513, 171, 264, 1024, HANDWRITTEN), (1000, 500, 3072, 1024, HANDWRITTEN),
    (1281, 700, 264, 64, HANDWRITTEN), (1300, 650, 3072, 3072, HANDWRITTEN), (1536, 512, 3072, 3072, HANDWRITTEN), (1100, 100, 520, 8192, HANDWRITTEN),
    (130, 65, 72, 256, 0), (1300, 650, 3072, 3072, 0),
])
def test_gates_for_groups_of_rows(gpu, M, rows, N, K, flags):
    from vllm_omni_amd import kernels

    x, w, residual, _, _, out = _operands(gpu, M, N, K)
    groups = -(-M // rows)
    g = torch.Generator(device=gpu).manual_seed(M)
    gate, bias = 20 * torch.randn(groups, N, device=gpu, generator=g), torch.randn(groups, N, device=gpu, generator=g)
    stream = torch.cuda.current_stream().cuda_stream
    ws = kernels._linear_scratch(gpu.index or 0, stream)
    print(f"clip M={M} groups of {rows} N={N} K={K} flags={flags}", flush=True)

    def run(flags):
        out.zero_()
        _lib.check(_lib.load().odit_linear_rows(x.data_ptr(), w.data_ptr(), bias.data_ptr(), out.data_ptr(), residual.data_ptr(), gate.data_ptr(), M, N, K, K, K,
                                                N, N, PRE, 2, 1, rows, N, flags, ws.data_ptr(), ws.numel(), stream), "odit_linear_rows")
        return out.clone()

    plain, got = run(flags), run(flags | CLIP)
    _same(got, plain)
    exact = residual.double() + (x.double() @ w.double().t()) * gate.double().repeat_interleave(rows, 0)[:M] + bias.double().repeat_interleave(rows, 0)[:M]
    there = ~exact.isnan()  # (each group its own gate: a rounding of the result, and 2^-18 of what is added up)
    assert bool(((got.double() - exact.clamp(-65504, 65504))[there].abs() <= 2.0 ** -10 * exact[there].abs().clamp(max=65504) + 2.0 ** -18 * 100 * 20 * K ** 0.5 * 0.05 + 1e-2).all())


@pytest.mark.parametrize("rows, entries, N, K", [((660, 180), 2, 1024, 1024), ((2200, 66), 2, 3072, 3072), ((140, 40), 2, 256, 256)])
def test_two_projections_with_gates_per_entry(gpu, rows, entries, N, K):
    from vllm_omni_amd import kernels

    ops = [_operands(gpu, m, N, K) for m in rows]
    g = torch.Generator(device=gpu).manual_seed(N)
    q, held = (_lib.LinearProblem * 2)(), []
    for i, (x, w, residual, _, _, out) in enumerate(ops):
        held.append((20 * torch.randn(entries, N, device=gpu, generator=g), torch.randn(entries, N, device=gpu, generator=g)))
        q[i].x, q[i].w, q[i].bias, q[i].residual, q[i].gate, q[i].out, q[i].M = (*(t.data_ptr() for t in (x, w, held[i][1], residual, held[i][0], out)), rows[i])
        q[i].ldx = q[i].ldw = K
        q[i].ldo = q[i].ldr = q[i].gate_stride = N
        q[i].rows_per_gate = rows[i] // entries
    stream = torch.cuda.current_stream().cuda_stream
    ws = kernels._linear_scratch(gpu.index or 0, stream)
    print(f"clip rows={rows} in {entries} entries N={N} K={K}", flush=True)

    def run(flags):
        _lib.check(_lib.load().odit_linear_pair(C.addressof(q), N, K, PRE, 2, 1, flags, ws.data_ptr(), ws.numel(), stream), "odit_linear_pair")
        return [o[-1].clone() for o in ops]

    plain, got = run(0), run(CLIP2)
    _same(got[1], plain[1])
    assert torch.equal(got[0].nan_to_num(7.0, 9.0, -9.0), plain[0].nan_to_num(7.0, 9.0, -9.0)), "the first problem's rows are as they come"
    _same(run(CLIP)[0], plain[0])
