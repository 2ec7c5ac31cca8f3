"""LayerNorm and modulation inside the launch of a small pair (odit_linear_pair_norm): the bits of the norm's own launch and the pair behind
it, for every number of steps, ragged rows and features, modulation rows per batch entry, plain outputs, GELU and heads of 64."""

import pytest
import torch

from vllm_omni_amd import _lib

pytestmark = pytest.mark.gpu

C = _lib.C


def _stream():
    return torch.cuda.current_stream().cuda_stream


class _Stream:
    """B entries of S rows of K features and what is done to them"""

    def __init__(self, gpu, dtype, B, S, K, N, heads, seed):
        g = torch.Generator(device=gpu).manual_seed(seed)

        def randn(*shape):
            return torch.randn(*shape, device=gpu, generator=g)

        self.B, self.S, self.K, self.N = B, S, K, N
        # rows far from zero mean, of unequal sizes, one of them constant
        self.x = (randn(B * S, K) * randn(B * S, 1).abs() + 3 * randn(B * S, 1)).to(dtype)
        self.x[B * S // 2] = 1.5
        self.mod = randn(B, 6 * K).to(dtype)
        self.w, self.b = (randn(N, K) * 0.05).to(dtype), randn(N).to(dtype)
        self.normed = torch.full_like(self.x, float("nan"))
        self.out = torch.full((B * S, N), float("nan"), dtype=dtype, device=gpu)
        if heads:
            self.wq, self.wk = (randn(64).mul(0.1).add(1).to(dtype) for _ in range(2))
            a = torch.rand(S, 32, device=gpu, generator=g) * 6.28
            self.cos, self.sin = a.cos().contiguous(), a.sin().contiguous()

    def problem(self, x):
        q = _lib.LinearProblem()
        q.x, q.w, q.bias, q.out, q.M = x.data_ptr(), self.w.data_ptr(), self.b.data_ptr(), self.out.data_ptr(), self.B * self.S
        q.ldx, q.ldw, q.ldo = self.K, self.K, self.N
        return q

    def norm(self):
        esz = 2
        return _lib.RowNorm(self.mod.data_ptr(), self.mod.data_ptr() + self.K * esz, 6 * self.K, self.S, 1e-6)

    def heads(self, joint, offset):
        h = _lib.HeadOutput()
        h.q, h.k, h.v = (t.data_ptr() for t in joint)
        h.wq, h.wk, h.cos, h.sin = self.wq.data_ptr(), self.wk.data_ptr(), self.cos.data_ptr(), self.sin.data_ptr()
        h.S, h.offset, h.S_total, h.H, h.D, h.eps = self.S, offset, joint[0].shape[1], self.N // 192, 64, 1e-6
        return h


def _normed(ps, hs, K, epilogue, code, launch=1, flags=0):
    q = (_lib.LinearProblem * 2)(*(p.problem(p.x) for p in ps))
    n = (_lib.RowNorm * 2)(*(p.norm() for p in ps))
    ptrs = (C.c_void_p * 2)(*(C.addressof(h) for h in hs)) if hs else None
    return _lib.load().odit_linear_pair_norm(C.addressof(q), C.addressof(n), ps[0].N, K, epilogue, ptrs, code, flags, launch, _stream())


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("heads", [False, True])
@pytest.mark.parametrize("B,S0,S1,K,N", [
    (1, 256, 64, 256, 768),   # the tiny model's
    (2, 65, 4, 64, 384),      # one step, entries of a few rows
    (3, 33, 20, 128, 192),    # two steps, tiles over several entries
    (1, 77, 130, 192, 192),   # three of four stages
    (2, 100, 31, 256, 960),   # tiles over two entries, ragged rows
])
def test_same_bits_as_the_norm_and_the_pair(gpu, dtype, heads, B, S0, S1, K, N):
    from vllm_omni_amd import kernels

    if not heads and N == 192:
        N = 200  # a ragged feature tile
    print(f"normed {dtype} heads={heads} B={B} {S0}+{S1} rows K={K} N={N}", flush=True)
    lib, code = _lib.load(), 0 if dtype == torch.bfloat16 else 1
    ws = kernels._linear_scratch(gpu.index or 0, _stream())
    ps = [_Stream(gpu, dtype, B, s, K, N, heads, 3 + i) for i, s in enumerate((S0, S1))]
    epilogues = (_lib.ODIT_EPI_BIAS,) if heads else (_lib.ODIT_EPI_BIAS, _lib.ODIT_EPI_BIAS_GELU_TANH)
    # the norm's own launch
    _lib.check(lib.odit_adaln_modulate_pair(
        _lib.ptr_array([p.x.data_ptr() for p in ps]), _lib.ptr_array([p.normed.data_ptr() for p in ps]), _lib.ptr_array([p.mod.data_ptr() for p in ps]),
        _lib.ptr_array([p.mod.data_ptr() + 2 * K for p in ps]), B, _lib.int_array([S0, S1]), K, _lib.i64_array([S0 * K, K, S1 * K, K]),
        _lib.i64_array([S0 * K, K, S1 * K, K]), _lib.i64_array([6 * K, 6 * K]), 1e-6, code, code, 0, _stream()), "odit_adaln_modulate_pair")
    for epilogue in epilogues:
        joint, want = ([torch.full((B, S0 + S1, N // 192, 64), float("nan"), dtype=dtype, device=gpu) for _ in range(3)] for _ in range(2))
        hs = [p.heads(joint, o) for p, o in zip(ps, (S1, 0))] if heads else None
        assert _normed(ps, hs, K, epilogue, code, launch=0) == 0 and all(bool(torch.isnan(p.out).all()) for p in ps)
        _lib.check(_normed(ps, hs, K, epilogue, code), "odit_linear_pair_norm")
        got = joint if heads else [p.out.clone() for p in ps]
        q = (_lib.LinearProblem * 2)(*(p.problem(p.normed) for p in ps))
        if heads:
            hw = [p.heads(want, o) for p, o in zip(ps, (S1, 0))]
            _lib.check(lib.odit_linear_heads(C.addressof(q), (C.c_int * 2)(N, N), K, (C.c_int * 2)(epilogue, epilogue),
                                             (C.c_void_p * 2)(*(C.addressof(h) for h in hw)), code, 0, 1, ws.data_ptr(), ws.numel(), _stream()), "odit_linear_heads")
        else:
            _lib.check(lib.odit_linear_pair(C.addressof(q), N, K, epilogue, code, code, 0, ws.data_ptr(), ws.numel(), _stream()), "odit_linear_pair")
            want = [p.out for p in ps]
        for a, b in zip(got, want):
            assert bool(torch.isfinite(b).all()) and torch.equal(a, b)
        for p in ps:
            p.out.fill_(float("nan"))


def test_what_it_leaves_to_the_calls_one_by_one(gpu):
    """More steps than stages, modulation rows off a 16-byte boundary, engines by name, more tiles than have a place: nothing launched."""
    code, dtype = 0, torch.bfloat16
    def pair(K, N=512, S=64):
        return [_Stream(gpu, dtype, 1, S, K, N, False, 9 + i) for i in range(2)]

    for ps, flags in ((pair(320), 0), (pair(256), _lib.ODIT_LINEAR_LIBRARY), (pair(256), _lib.ODIT_LINEAR_HANDWRITTEN), (pair(256), _lib.ODIT_LINEAR_NO_TILE),
                      (pair(256, N=4096, S=1024), 0)):
        assert _normed(ps, None, ps[0].K, _lib.ODIT_EPI_BIAS, code, flags=flags) == -2
        assert all(bool(torch.isnan(p.out).all()) for p in ps)
    ps = pair(256)
    ps[1].mod = torch.zeros(6 * 256 + 1, dtype=dtype, device=gpu)[1:].view(1, -1)
    assert _normed(ps, None, 256, _lib.ODIT_EPI_BIAS, code) == -2 and all(bool(torch.isnan(p.out).all()) for p in ps)
