"""Projections to query, key and value heads with the heads' norm and rotation at the tile's end (odit_linear_heads): what the two
projections in one launch of the tile kernel and the pass behind them give, and a float64 model of it; whole tiles and tiles cut along
the reduction, both tile heights, heads of 64 and 128 that begin anywhere in a tile, ragged rows, batch entries of few rows."""

import pytest
import torch

from vllm_omni_amd import _lib

pytestmark = pytest.mark.gpu

C = _lib.C
# rounding of the projection and of the result, 2^-9 / sqrt(3) * (1.33 on average over a binade) in the 2-norm each, and half as much again
_BOUND = {torch.bfloat16: 1.5 * 2 ** 0.5 * 1.7e-3, torch.float16: 1.5 * 2 ** 0.5 * 2.1e-4}


@pytest.fixture()
def scratch(gpu):
    from vllm_omni_amd import kernels

    ws = kernels._linear_scratch(gpu.index or 0, torch.cuda.current_stream().cuda_stream)
    yield ws
    assert int(ws[:32768].view(torch.int32).abs().max().item()) == 0, "ticket words are handed back at zero"


def _stream():
    return torch.cuda.current_stream().cuda_stream


class _Problem:
    """B entries of S rows, projected to N features; heads H of D, or a plain output where H is 0"""

    def __init__(self, gpu, dtype, B, S, K, H, D, N=0, seed=0, x=None):
        g = torch.Generator(device=gpu).manual_seed(seed)
        self.B, self.S, self.H, self.D, self.N = B, S, H, D, N or 3 * H * D
        self.x = x if x is not None else torch.randn(B * S, K, device=gpu, generator=g).to(dtype)
        self.w = (torch.randn(self.N, K, device=gpu, generator=g) * 0.05).to(dtype)
        self.b = torch.randn(self.N, device=gpu, generator=g).to(dtype)
        self.out = torch.full((B * S, self.N), float("nan"), dtype=dtype, device=gpu)
        if H:
            self.wq, self.wk = (torch.randn(D, device=gpu, generator=g).mul(0.1).add(1).to(dtype) for _ in range(2))
            a = torch.rand(S, D // 2, device=gpu, generator=g) * 6.28
            self.cos, self.sin = a.cos().contiguous(), a.sin().contiguous()

    def linear(self):
        q = _lib.LinearProblem()
        q.x, q.w, q.bias, q.out, q.M = self.x.data_ptr(), self.w.data_ptr(), self.b.data_ptr(), self.out.data_ptr(), self.B * self.S
        q.ldx, q.ldw, q.ldo = self.x.shape[1], self.x.shape[1], self.N
        return q

    def heads(self, joint, offset):
        h = _lib.HeadOutput()
        h.q, h.k, h.v = (t.data_ptr() for t in joint)
        h.wq, h.wk, h.cos, h.sin = self.wq.data_ptr(), self.wk.data_ptr(), self.cos.data_ptr(), self.sin.data_ptr()
        h.S, h.offset, h.S_total, h.H, h.D, h.eps = self.S, offset, joint[0].shape[1], self.H, self.D, 1e-6
        return h

    def model(self):
        """float64 of the projection as it is stored: q, k, v [B, S, H, D]"""
        y = (self.x.double() @ self.w.double().t() + self.b.double()).to(self.x.dtype).double().view(self.B, self.S, 3, self.H, self.D)
        res = []
        for i, w in ((0, self.wq), (1, self.wk)):
            n = y[:, :, i] * torch.rsqrt(y[:, :, i].pow(2).mean(-1, keepdim=True) + 1e-6) * w.double()
            c, s = self.cos.double()[None, :, None, :], self.sin.double()[None, :, None, :]
            a, b = n[..., 0::2], n[..., 1::2]
            res.append(torch.stack((a * c - b * s, b * c + a * s), -1).flatten(-2))
        return res + [y[:, :, 2]]


def _run(ps, offsets, joint, K, dtype, ws, epilogue=(1, 1), launch=1, flags=0, plain=-1):
    """`plain`: the problem of this number as an ordinary projection, into its `out`."""
    q = (_lib.LinearProblem * 2)(*(p.linear() for p in ps))
    hs = [p.heads(joint, o) if p.H and i != plain else None for i, (p, o) in enumerate(zip(ps, offsets))]
    ptrs = (C.c_void_p * 2)(*(C.addressof(h) if h is not None else None for h in hs))
    return _lib.load().odit_linear_heads(C.addressof(q), (C.c_int * 2)(ps[0].N, ps[1].N), K, (C.c_int * 2)(*epilogue), ptrs,
                                         0 if dtype == torch.bfloat16 else 1, flags, launch, ws.data_ptr(), ws.numel(), _stream())


def _check(ps, offsets, joint, dtype):
    for p, o in zip(ps, offsets):
        if p.H:
            for got, want in zip(joint, p.model()):
                part = got[:, o:o + p.S].double().view_as(want)
                assert torch.isfinite(part).all()
                assert ((part - want).norm() / want.norm()).item() < _BOUND[dtype]
                # and of every pair that is rotated together: the projection falls on the neighbour of the model's value at worst (2 u), which
                # the rotation leaves its length, and the result is rounded once (u); float32 sums of a head's scale on top
                u = torch.finfo(dtype).eps / 2
                pairs, rms = want.unflatten(-1, (-1, 2)).norm(dim=-1), want.pow(2).mean(-1, keepdim=True).sqrt()
                assert bool(((part - want).unflatten(-1, (-1, 2)).norm(dim=-1) <= 3.1 * u * pairs + 2e-5 * rms).all())


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("B,S0,S1,H,D,K", [
    (2, 1024, 171, 24, 128, 3072),  # 256-row tiles, the last round's in two parts
    (1, 1021, 509, 9, 128, 1024),   # ragged rows, an odd number of heads
    (2, 256, 40, 24, 128, 3072),    # 128-row tiles
    (1, 700, 77, 15, 64, 4096),     # heads of 64 that end in the middle of a half tile, parts
    (3, 531, 9, 10, 64, 512),       # batch entries of a few rows
    (130, 8, 1, 8, 128, 1024),      # one row to a batch entry
    (1, 2300, 300, 8, 128, 8192),   # three and four parts
])
def test_heads_of_two_streams(scratch, gpu, dtype, B, S0, S1, H, D, K):
    print(f"heads {dtype} B={B} {S0}+{S1} rows, {H} x {D}, K={K}", flush=True)
    ps = [_Problem(gpu, dtype, B, S0, K, H, D, seed=1), _Problem(gpu, dtype, B, S1, K, H, D, seed=2)]
    joint = [torch.full((B, S0 + S1, H, D), float("nan"), dtype=dtype, device=gpu) for _ in range(3)]
    force = _lib.ODIT_LINEAR_HANDWRITTEN
    assert _run(ps, (S1, 0), joint, K, dtype, scratch, launch=0, flags=force) == 0 and all(torch.isnan(t).all() for t in joint)
    _lib.check(_run(ps, (S1, 0), joint, K, dtype, scratch, flags=force), "odit_linear_heads")
    _check(ps, (S1, 0), joint, dtype)
    first = [t.clone() for t in joint]
    for _ in range(3):
        _lib.check(_run(ps, (S1, 0), joint, K, dtype, scratch, flags=force), "odit_linear_heads")
        assert all(torch.equal(a, b) for a, b in zip(first, joint))
    # the projections as ordinary ones, each beside the other's heads in a launch that is laid out the same way, and the pass: the same bits
    lib, code = _lib.load(), 0 if dtype == torch.bfloat16 else 1
    for i in range(2):
        _lib.check(_run(ps, (S1, 0), [torch.empty_like(t) for t in joint], K, dtype, scratch, flags=force, plain=i), "odit_linear_heads")
        assert bool(torch.isfinite(ps[i].out).all())
    want = [torch.full_like(t, float("nan")) for t in joint]
    esz, HD = 2, H * D
    for p, o in zip(ps, (S1, 0)):
        at = p.out.data_ptr()
        _lib.check(lib.odit_qknorm_rope(at, at + HD * esz, at + 2 * HD * esz, *(t.data_ptr() for t in want), p.wq.data_ptr(), p.wk.data_ptr(), p.cos.data_ptr(),
                                        p.sin.data_ptr(), B, p.S, H, D, D, _lib.i64_array([p.S * 3 * HD, 3 * HD]), o, S0 + S1, 1e-6, _lib.ODIT_NORM_HEAD, code,
                                        code, 0, _stream()), "odit_qknorm_rope")
    assert torch.equal(want[2], joint[2])
    for a, b in zip(want[:2], joint[:2]):  # (an odd feature is a sum of two products, of which the compiler rounds one or the other)
        assert torch.equal(a[..., 0::2], b[..., 0::2])
        assert (a != b).float().mean().item() < 1e-3 and ((a.double() - b.double()).norm() / a.double().norm()).item() < 1e-4


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("B,S,H,D,N,K", [
    (1, 1536, 24, 128, 12288, 3072),  # two rounds of whole tiles
    (2, 555, 5, 64, 5000, 1024),      # ragged
    (1, 512, 16, 128, 4096, 5120),    # parts of either problem
])
def test_heads_beside_a_gelu_projection(scratch, gpu, dtype, B, S, H, D, N, K):
    plain = _Problem(gpu, dtype, B, S, K, 0, 0, N=N, seed=3)
    ps = [plain, _Problem(gpu, dtype, B, S, K, H, D, seed=4, x=plain.x)]
    joint = [torch.full((B, S, H, D), float("nan"), dtype=dtype, device=gpu) for _ in range(3)]
    _lib.check(_run(ps, (0, 0), joint, K, dtype, scratch, epilogue=(3, 1), flags=_lib.ODIT_LINEAR_HANDWRITTEN), "odit_linear_heads")
    _check(ps, (0, 0), joint, dtype)
    want = torch.nn.functional.gelu(plain.x.double() @ plain.w.double().t() + plain.b.double(), approximate="tanh")
    assert ((plain.out.double() - want).norm() / want.norm()).item() < _BOUND[dtype]
    assert _run(ps, (0, 0), joint, K, dtype, scratch, epilogue=(3, 1), flags=_lib.ODIT_LINEAR_LIBRARY) == -2  # ODIT_ENOTSUP
    assert _run(ps, (0, 0), joint, K, dtype, scratch, epilogue=(3, 1), flags=_lib.ODIT_LINEAR_NO_TILE) == -2


def test_rows_that_do_not_fit_are_refused(scratch, gpu):
    ps = [_Problem(gpu, torch.bfloat16, 1, 300, 1024, 8, 128, seed=5), _Problem(gpu, torch.bfloat16, 1, 40, 1024, 8, 128, seed=6)]
    joint = [torch.full((1, 339, 8, 128), float("nan"), dtype=torch.bfloat16, device=gpu) for _ in range(3)]
    assert _run(ps, (40, 0), joint, 1024, torch.bfloat16, scratch) == -1  # ODIT_EINVAL
    assert all(torch.isnan(t).all() for t in joint)


def test_heads_in_one_launch_where_that_is_expected_to_be_faster(scratch, gpu):
    """Many rows take the pass with the projections; 512 + 80 rows run on the stream-K kernel, whose time the tile kernel does not reach."""
    for S0, S1, want in ((1024, 256, 0), (256, 40, -2)):
        ps = [_Problem(gpu, torch.bfloat16, 2, S, 3072, 24, 128, seed=S) for S in (S0, S1)]
        joint = [torch.empty(2, S0 + S1, 24, 128, dtype=torch.bfloat16, device=gpu) for _ in range(3)]
        assert _run(ps, (S1, 0), joint, 3072, torch.bfloat16, scratch, launch=0) == want


def test_what_was_answered_is_launched(scratch, gpu):
    """A caller that has laid its memory out by an answer gets the launch, whatever is expected by then; operands are checked as ever."""
    ps = [_Problem(gpu, torch.bfloat16, 2, S, 3072, 24, 128, seed=S) for S in (256, 40)]
    joint = [torch.full((2, 296, 24, 128), float("nan"), dtype=torch.bfloat16, device=gpu) for _ in range(3)]
    assert _run(ps, (40, 0), joint, 3072, torch.bfloat16, scratch, launch=_lib.ODIT_LAUNCH_CHOOSE) == -2  # ODIT_ENOTSUP
    assert all(bool(t.isnan().all()) for t in joint)
    assert _run(ps, (40, 0), joint, 3072, torch.bfloat16, scratch, launch=_lib.ODIT_LAUNCH_ANSWERED) == 0
    _check(ps, (40, 0), joint, torch.bfloat16)
    assert _run(ps, (41, 0), joint, 3072, torch.bfloat16, scratch, launch=_lib.ODIT_LAUNCH_ANSWERED) == -1  # ODIT_EINVAL: rows past the joint tensors
    assert _run(ps, (40, 0), joint, 3072, torch.bfloat16, scratch, launch=_lib.ODIT_LAUNCH_ANSWERED, flags=_lib.ODIT_LINEAR_LIBRARY) == -2


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("B,S0,S1,H,K", [
    (1, 256, 64, 4, 256),   # whole tiles
    (2, 75, 9, 4, 64),      # one step, batch entries that end inside a tile
    (3, 100, 5, 3, 128),    # an odd number of heads
    (1, 8, 65, 5, 512),     # fewer rows than a tile, one row more
    (33, 1, 2, 2, 1024),    # batch entries of one and two rows, more steps than stages
])
def test_heads_of_small_products(scratch, gpu, dtype, B, S0, S1, H, K):
    """The small kernel, whose tile is a head of 64: the bits of its pair launch and the pass behind it."""
    print(f"small heads {dtype} B={B} {S0}+{S1} rows, {H} x 64, K={K}", flush=True)
    ps = [_Problem(gpu, dtype, B, S0, K, H, 64, seed=7), _Problem(gpu, dtype, B, S1, K, H, 64, seed=8)]
    joint = [torch.full((B, S0 + S1, H, 64), float("nan"), dtype=dtype, device=gpu) for _ in range(3)]
    _lib.check(_run(ps, (S1, 0), joint, K, dtype, scratch), "odit_linear_heads")
    _check(ps, (S1, 0), joint, dtype)
    lib, code = _lib.load(), 0 if dtype == torch.bfloat16 else 1
    q = (_lib.LinearProblem * 2)(*(p.linear() for p in ps))
    N = 3 * H * 64
    _lib.check(lib.odit_linear_pair(C.addressof(q), N, K, 1, code, code, 0, scratch.data_ptr(), scratch.numel(), _stream()), "odit_linear_pair")
    want = [torch.full_like(t, float("nan")) for t in joint]
    for p, o in zip(ps, (S1, 0)):
        at = p.out.data_ptr()
        _lib.check(lib.odit_qknorm_rope(at, at + H * 128, at + H * 256, *(t.data_ptr() for t in want), p.wq.data_ptr(), p.wk.data_ptr(), p.cos.data_ptr(),
                                        p.sin.data_ptr(), B, p.S, H, 64, 64, _lib.i64_array([p.S * N, N]), o, S0 + S1, 1e-6, _lib.ODIT_NORM_HEAD, code, code, 0,
                                        _stream()), "odit_qknorm_rope")
    assert torch.equal(want[2], joint[2])
    for a, b in zip(want[:2], joint[:2]):
        assert torch.equal(a[..., 0::2], b[..., 0::2])
        assert (a != b).float().mean().item() < 1e-3 and ((a.double() - b.double()).norm() / a.double().norm()).item() < 1e-4
