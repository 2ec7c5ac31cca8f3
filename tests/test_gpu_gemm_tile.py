"""The tile kernel (csrc/gemm_tile.h) where it can go wrong: whole tiles, tiles cut along the reduction into 2, 3 and 4
parts, alone and behind whole rounds, ragged edges, two problems in one launch, ticket words left behind, graph replays.

The reference is a float64 product. A result is one rounding of an fp32 sum: its relative error in the 2-norm is that of the
rounding, 2^-9 / sqrt(3) * (1.33 on average over a binade) = 1.7e-3 in bf16 and an eighth of it in fp16; the fp32 sums add less
than 1e-5. Bound: 1.5 times that."""

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


def _gelu(y):
    return torch.nn.functional.gelu(y, approximate="tanh")


@pytest.fixture()
def kernels(gpu):
    from vllm_omni_amd import kernels as k

    yield k
    for ws in k._LINEAR_SCRATCH.values():
        assert int(ws[:32768].view(torch.int32).abs().max().item()) == 0, "ticket words are handed back at zero"


_SHAPES = [
    (1100, 200, 192),     # 128 x 256 tiles, ragged both ways, three steps
    (1025, 8, 64),        # one step, one feature group, one row in the last tile
    (1100, 1000, 2048),   # 128 x 256 tiles in 4 parts
    (1100, 2056, 2048),   # 3 parts, one feature group in the last tile
    (1100, 3080, 8192),   # 2 parts
    (1300, 3072, 6144),   # 256 x 256 tiles in 3 parts
    (1100, 3072, 8192),   # 4 parts
    (1100, 5128, 8192),   # 2 parts
    (1280, 12296, 512),   # a round of whole 256 x 256 tiles
    (4200, 4104, 4096),   # a round of whole tiles behind 33 tiles in 4 parts
    (4200, 4104, 192),    # two rounds, the second of 33 tiles
]


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("M,N,K", _SHAPES)
def test_tile_gemm(kernels, gpu, dtype, M, N, K):
    x, w, b, y = _mk(gpu, M, N, K, dtype, M + N + K)
    print(f"tile kernel {dtype} {M}x{N}x{K}", flush=True)
    first = kernels.linear(x, w, b, engine="handwritten")
    assert _rel(first, y + b.double()) < _BOUND[dtype]
    for _ in range(3):  # (the order of the partial sums does not depend on who arrives last)
        assert torch.equal(first, kernels.linear(x, w, b, engine="handwritten"))
    assert _rel(kernels.linear(x, w, b, activation="gelu_tanh", engine="handwritten"), _gelu(y + b.double())) < _BOUND[dtype]
    S = M // 2  # groups of rows end inside a tile, the last one has one row where M is odd
    groups = -(-M // S)
    g = torch.Generator(device=gpu).manual_seed(3)
    gate = torch.randn(groups, N, device=gpu, generator=g)
    if M % S == 0:
        h = torch.randn(groups, S, N, device=gpu, generator=g).to(dtype)
        want = h.double() + gate.double()[:, None, :] * (y + b.double()).view(groups, S, N)
        got = kernels.linear(x.view(groups, S, K), w, None, residual=h, gate=gate, gate_bias=gate * b.float(), prescaled=True, engine="handwritten")
        assert _rel(got, want) < _BOUND[dtype]
        kernels.linear(x.view(groups, S, K), w, None, residual=h, gate=gate, gate_bias=gate * b.float(), prescaled=True, out=h, engine="handwritten")
        assert torch.equal(h, got), "in place"


def _pair(lib, ws, q, N, K, epilogue, code, flags=0):
    from vllm_omni_amd import _lib

    rc = lib.odit_linear_pair(_lib.C.addressof(q), N, K, epilogue, 2, code, flags, ws.data_ptr(), ws.numel(),
                              torch.cuda.current_stream().cuda_stream)
    return rc


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("M0,M1,N,K", [
    (1024, 512, 9216, 3072),   # whole 256-row tiles of both
    (1021, 511, 9208, 3072),   # ragged
    (2048, 342, 3072, 12288),  # tiles in 2 parts, those of the second problem among them
    (1024, 512, 3072, 12288),  # 3 parts
    (2048, 342, 3072, 3072),   # 128-row tiles
])
def test_tile_gemm_pair(kernels, gpu, dtype, M0, M1, N, K):
    """Two problems in one launch: bias, GELU, and gates per group of rows."""
    from vllm_omni_amd import _lib

    lib, code = _lib.load(), 0 if dtype == torch.bfloat16 else 1
    ws = kernels._linear_scratch(gpu.index or 0, torch.cuda.current_stream().cuda_stream)
    ops = [_mk(gpu, m, N, K, dtype, m + i) for i, m in enumerate((M0, M1))]
    g = torch.Generator(device=gpu).manual_seed(9)
    res = [torch.randn(m, N, device=gpu, generator=g).to(dtype) for m in (M0, M1)]
    rows = [max(1, m // 2) for m in (M0, M1)]
    gates = [torch.randn(-(-m // r), N, device=gpu, generator=g) for m, r in zip((M0, M1), rows)]
    scaled = [t * o[2].float() for t, o in zip(gates, ops)]
    out = [torch.full((m, N), float("nan"), dtype=dtype, device=gpu) for m in (M0, M1)]

    def run(epilogue):
        q = (_lib.LinearProblem * 2)()
        for i, m in enumerate((M0, M1)):
            q[i].x, q[i].w, q[i].bias, q[i].out, q[i].M = ops[i][0].data_ptr(), ops[i][1].data_ptr(), ops[i][2].data_ptr(), out[i].data_ptr(), m
            q[i].ldx, q[i].ldw, q[i].ldo, q[i].ldr = K, K, N, N
            if epilogue == 5:
                q[i].bias, q[i].residual, q[i].gate = scaled[i].data_ptr(), res[i].data_ptr(), gates[i].data_ptr()
                q[i].rows_per_gate, q[i].gate_stride = rows[i], N
        _lib.check(_pair(lib, ws, q, N, K, epilogue, code), "odit_linear_pair")
        return [t.clone() for t in out]

    plain = [o[3] + o[2].double() for o in ops]
    got = run(1)
    assert all(_rel(a, b) < _BOUND[dtype] for a, b in zip(got, plain))
    assert all(torch.equal(a, b) for a, b in zip(got, run(1)))
    assert all(_rel(a, _gelu(b)) < _BOUND[dtype] for a, b in zip(run(3), plain))
    per_row = [t[torch.arange(m, device=gpu) // r].double() for t, m, r in zip(gates, (M0, M1), rows)]
    want = [r.double() + p * y for r, p, y in zip(res, per_row, plain)]
    assert all(_rel(a, b) < _BOUND[dtype] for a, b in zip(run(5), want))


def test_tile_gemm_overrides_stale_ticket_words(kernels, gpu):
    """Words as a launch that never finished would leave them (arrivals, given-up quadrants and departures of an old epoch)."""
    M, N, K = 1100, 1000, 2048
    x, w, b, _ = _mk(gpu, M, N, K, torch.bfloat16, 1)
    want = kernels.linear(x, w, b, engine="handwritten")
    ws = kernels._linear_scratch(gpu.index or 0, torch.cuda.current_stream().cuda_stream)
    with torch.inference_mode():  # (the scratch may have been made there)
        ws[:32768].view(torch.int64).fill_((1 << 16) | 0x3F3)
        assert torch.equal(kernels.linear(x, w, b, engine="handwritten"), want)
        ws[:32768].zero_()  # words of tiles that this problem does not have


@pytest.mark.parametrize("M,N,K", [(1100, 1000, 2048), (1100, 2056, 2048), (1100, 5128, 8192), (4200, 4104, 4096)])
def test_parts_that_do_not_run_at_once(kernels, gpu, M, N, K):
    """Cut tiles while two other streams keep the compute units busy: parts start long after each other, so some give their
    quadrants up to the last one. The sums are formed in one order whoever forms them: the same bits as alone."""
    x, w, b, _ = _mk(gpu, M, N, K, torch.bfloat16, 3)
    want = kernels.linear(x, w, b, engine="handwritten")
    here, others = torch.cuda.current_stream(), [torch.cuda.Stream() for _ in range(2)]
    busy = [torch.randn(4096, 4096, device=gpu).bfloat16() for _ in range(2)]
    torch.cuda.synchronize()
    outs = []
    for s, t in zip(others, busy):
        with torch.cuda.stream(s):
            for _ in range(12):
                kernels.linear(t, t, None, engine="handwritten")
    for _ in range(12):
        outs.append(kernels.linear(x, w, b, engine="handwritten"))
    for s in others:
        here.wait_stream(s)
    torch.cuda.synchronize()
    assert all(torch.equal(o, want) for o in outs)


def test_tile_gemm_in_a_graph(kernels, gpu):
    """Cut tiles under capture: every replay gives the eager result, with eager launches in between."""
    M, N, K = 1100, 2056, 2048
    x, w, b, _ = _mk(gpu, M, N, K, torch.bfloat16, 2)
    want = kernels.linear(x, w, b, engine="handwritten")
    out, side = torch.empty_like(want), torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        kernels.linear(x, w, b, out=out, engine="handwritten")
    torch.cuda.current_stream().wait_stream(side)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        kernels.linear(x, w, b, out=out, engine="handwritten")
    for _ in range(4):
        out.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, want)
        assert torch.equal(kernels.linear(x, w, b, engine="handwritten"), want)
    del graph


def test_pair_of_tuned_problems_is_one_launch_where_that_is_faster(kernels, gpu):
    """Tuning records for one and for both problems: one launch (30 us) stays the choice against two calls, of 26 and 17 us as
    tuned and of 28 and 20 as expected."""
    from vllm_omni_amd import _lib

    M0, M1, N, K = 1216, 448, 6144, 1024  # (sizes that no other test tunes)
    lib = _lib.load()
    ws = kernels._linear_scratch(gpu.index or 0, torch.cuda.current_stream().cuda_stream)
    ops = [_mk(gpu, m, N, K, torch.bfloat16, m) for m in (M0, M1)]
    out = [torch.empty(m, N, dtype=torch.bfloat16, device=gpu) for m in (M0, M1)]
    q = (_lib.LinearProblem * 2)()
    for i, m in enumerate((M0, M1)):
        q[i].x, q[i].w, q[i].bias, q[i].out, q[i].M = ops[i][0].data_ptr(), ops[i][1].data_ptr(), ops[i][2].data_ptr(), out[i].data_ptr(), m
        q[i].ldx, q[i].ldw, q[i].ldo, q[i].ldr = K, K, N, N
    assert _pair(lib, ws, q, N, K, 1, 0) == 0
    for (x, w, b, _), o in zip(ops, out):
        kernels.linear(x, w, b, out=o, tune_iters=2)
        assert _pair(lib, ws, q, N, K, 1, 0) == 0


def test_pair_that_is_two_calls_stays_two_calls_when_tuned(kernels, gpu):
    """Two calls take 103 us, one launch 106. What a tuning call measures behind its cache flush is longer than a call in a model."""
    from vllm_omni_amd import _lib

    M0, M1, N, K = 1122, 185, 12288, 3072
    lib = _lib.load()
    ws = kernels._linear_scratch(gpu.index or 0, torch.cuda.current_stream().cuda_stream)
    q, ops = (_lib.LinearProblem * 2)(), []
    for i, m in enumerate((M0, M1)):
        x, w, b, _ = _mk(gpu, m, N, K, torch.bfloat16, m)
        out = torch.empty(m, N, dtype=torch.bfloat16, device=gpu)
        q[i].x, q[i].w, q[i].bias, q[i].out, q[i].M = x.data_ptr(), w.data_ptr(), b.data_ptr(), out.data_ptr(), m
        q[i].ldx, q[i].ldw, q[i].ldo, q[i].ldr = K, K, N, N
        ops.append((x, w, b, out))
    assert _pair(lib, ws, q, N, K, 1, 0) == -2  # ODIT_ENOTSUP
    for x, w, b, out in ops:
        kernels.linear(x, w, b, out=out, tune_iters=3)
        assert _pair(lib, ws, q, N, K, 1, 0) == -2


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("M,N0,N1,K", [
    (1536, 12288, 9216, 3072),  # two rounds of whole 256-row tiles
    (1111, 5000, 4104, 1024),   # ragged rows and features of both
    (512, 5120, 5120, 5120),    # tiles in parts, those of either problem
])
def test_tile_gemm_fork(kernels, gpu, dtype, M, N0, N1, K):
    """One x, two weights of different widths, GELU on the first."""
    from vllm_omni_amd import _lib

    lib, code, C = _lib.load(), 0 if dtype == torch.bfloat16 else 1, _lib.C
    ws = kernels._linear_scratch(gpu.index or 0, torch.cuda.current_stream().cuda_stream)
    x, w0, b0, y0 = _mk(gpu, M, N0, K, dtype, 21)
    _, w1, b1, _ = _mk(gpu, 8, N1, K, dtype, 22)
    y1 = x.double() @ w1.double().t()
    out = [torch.full((M, n), float("nan"), dtype=dtype, device=gpu) for n in (N0, N1)]
    q = (_lib.LinearProblem * 2)()
    for i, (w, b, n) in enumerate(((w0, b0, N0), (w1, b1, N1))):
        q[i].x, q[i].w, q[i].bias, q[i].out, q[i].M = x.data_ptr(), w.data_ptr(), b.data_ptr(), out[i].data_ptr(), M
        q[i].ldx, q[i].ldw, q[i].ldo = K, K, n

    def run(flags):
        return lib.odit_linear_fork(C.addressof(q), (C.c_int * 2)(N0, N1), K, (C.c_int * 2)(3, 1), code, flags, ws.data_ptr(), ws.numel(),
                                    torch.cuda.current_stream().cuda_stream)

    assert run(_lib.ODIT_LINEAR_LIBRARY) == run(_lib.ODIT_LINEAR_NO_TILE) == -2  # ODIT_ENOTSUP
    _lib.check(run(0), "odit_linear_fork")
    assert _rel(out[0], _gelu(y0 + b0.double())) < _BOUND[dtype] and _rel(out[1], y1 + b1.double()) < _BOUND[dtype]
    first = [t.clone() for t in out]
    for _ in range(3):
        _lib.check(run(0), "odit_linear_fork")
        assert all(torch.equal(a, b) for a, b in zip(first, out))


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("B,S,N,K,K2", [
    (1, 1536, 3072, 3072, 12288),  # 3 parts: the sources change inside a part
    (2, 700, 3072, 3072, 12288),   # gate vectors change inside a tile
    (1, 4608, 3072, 3072, 12288),  # a round of whole tiles
    (1, 1100, 1032, 64, 8192),     # one step of the first source, ragged
    (2, 640, 2048, 8192, 64),      # one step of the second
])
def test_tile_gemm_join(kernels, gpu, dtype, B, S, N, K, K2):
    """Rows in two tensors as one reduction, gated, in place and not."""
    from vllm_omni_amd import _lib

    lib, code, M = _lib.load(), 0 if dtype == torch.bfloat16 else 1, B * S
    ws = kernels._linear_scratch(gpu.index or 0, torch.cuda.current_stream().cuda_stream)
    x, w, b, _ = _mk(gpu, M, N, K + K2, dtype, 31)
    xa, xb = x[:, :K].contiguous(), x[:, K:].contiguous()
    g = torch.Generator(device=gpu).manual_seed(32)
    h, gate = torch.randn(M, N, device=gpu, generator=g).to(dtype), torch.randn(B, N, device=gpu, generator=g)
    gb = gate * b.float()
    rows = torch.arange(M, device=gpu) // S
    want = h.double() + gate.double()[rows] * (x.double() @ w.double().t()) + gb.double()[rows]

    def run(res, out, flags=0):
        return lib.odit_linear_join(xa.data_ptr(), xb.data_ptr(), w.data_ptr(), gb.data_ptr(), out.data_ptr(), res.data_ptr(), gate.data_ptr(),
                                    M, N, K, K2, K, K2, K + K2, N, N, 5, 2, code, S if B > 1 else 0, N, flags, ws.data_ptr(), ws.numel(),
                                    torch.cuda.current_stream().cuda_stream)

    out = torch.full_like(h, float("nan"))
    assert run(h, out, _lib.ODIT_LINEAR_LIBRARY) == -2  # ODIT_ENOTSUP
    _lib.check(run(h, out), "odit_linear_join")
    assert _rel(out, want) < _BOUND[dtype]
    for _ in range(3):
        again = h.clone()
        _lib.check(run(again, again), "odit_linear_join")
        assert torch.equal(again, out)
