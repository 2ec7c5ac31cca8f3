"""A timestep per token (``odit_time_tokens``): rows of distinct timesteps formed once where there are at most four, all of them otherwise."""

import pytest
import torch

from vllm_omni_amd import _lib, kernels
from vllm_omni_amd.blocks.qwen_image import QwenTimestepProjEmbeddings, TimestepEmbedding

pytestmark = pytest.mark.gpu
BF16, F16, F32 = torch.bfloat16, torch.float16, torch.float32


def _modules(gpu, dtype, C, P, bias=True):
    emb, proj = TimestepEmbedding(256, C).to(device=gpu, dtype=dtype), torch.nn.Linear(C, P, bias=bias, device=gpu, dtype=dtype)
    with torch.no_grad():
        for lin in (emb.linear_1, emb.linear_2, proj):
            lin.weight.normal_(0, lin.in_features ** -0.5)
    return emb, proj


def _spread(done):
    return done if done is None else tuple(x[done[2].long()] for x in done[:2])


def _as_before(emb, proj, t, dtype):
    temb = emb(QwenTimestepProjEmbeddings.time_proj(t, scale=1.0, dtype=dtype))
    return temb, kernels.project(proj, temb, silu_input=True)


def _in_double(emb, proj, t, dtype):
    """With the roundings to the type that every step has."""
    def lin(m, x):
        return (x.double() @ m.weight.double().t() + (m.bias.double() if m.bias is not None else 0)).to(dtype)

    def silu(x):
        return torch.nn.functional.silu(x.double()).to(dtype)
    temb = lin(emb.linear_2, silu(lin(emb.linear_1, QwenTimestepProjEmbeddings.time_proj(t, scale=1.0, dtype=dtype))))
    return temb, lin(proj, silu(temb))


# C a multiple of 512: the stream kernel's rows; others the matrix kernel's. 8192 and more tokens: more than one trip of the search
@pytest.mark.parametrize("n,C,P", [(2706, 1536, 9216), (1100, 1024, 6144), (8193, 1088, 2176), (20000, 512, 3072)])
@pytest.mark.parametrize("dtype,t_dtype,bias", [(BF16, F32, True), (F16, BF16, False)])
@pytest.mark.parametrize("distinct", [1, 2, 3, 4, 5, 9])
def test_distinct_timesteps(gpu, n, C, P, dtype, t_dtype, bias, distinct):
    print(f"timesteps of {n} tokens, {distinct} distinct, {C} {P} {dtype}", flush=True)
    torch.manual_seed(n + distinct)
    emb, proj = _modules(gpu, dtype, C, P, bias)
    values = (torch.randperm(900, device=gpu)[:distinct].to(t_dtype) if t_dtype == F32 else torch.arange(distinct, device=gpu).to(t_dtype) * 8)
    t = values[torch.randint(distinct, (n,), device=gpu)]
    t[:distinct] = values.flip(0)
    t[n - 1] = values[0]  # (the last one alone may be the one of its kind)
    with torch.inference_mode():
        done = kernels.time_tokens(emb, proj, t, 256, 10000, 1.0, dtype)
        got = _spread(done)
        assert done[2].dtype == torch.int32 and (torch.equal(done[2].long(), torch.arange(n, device=gpu)) if distinct > 4 else
                                                 int(done[2].min()) == 0 and int(done[2].max()) == distinct - 1)
        before = _as_before(emb, proj, t, dtype)
        for a, b in zip(got, before, strict=True):
            # (of more distinct ones the same rows in tiles that are cut along the reduction and in whole ones differ by their order)
            assert a.shape == b.shape and all(distinct > 4 or int(torch.unique(a[t == v], dim=0).shape[0]) == 1 for v in values)
        # beside 64-bit sums only the elements differ whose float32 sum rounds to the type the other way, a step apart, and what follows from
        # them: less in all than a row of which every element is a step off
        tol = 2.0 ** -8 if dtype == BF16 else 2.0 ** -11
        for a, b, w in zip(got, before, _in_double(emb, proj, values, dtype), strict=True):
            for v, row in zip(values, w.double()):
                i = int((t == v).nonzero()[0])
                for x in (a, b):
                    assert float((x[i].double() - row).norm() / row.norm()) < tol


def test_bit_patterns(gpu):
    """Infinities and NaN are timesteps like others; zeros of both signs give the same rows."""
    emb, proj = _modules(gpu, BF16, 1536, 9216)
    t = torch.tensor([0.0, -0.0, 700.0, 0.0], device=gpu).repeat(700)
    with torch.inference_mode():
        temb, rows = _spread(kernels.time_tokens(emb, proj, t, 256, 10000, 1.0, BF16))
        assert torch.equal(temb[0], temb[1]) and torch.equal(rows[0], rows[1]) and not torch.equal(temb[0], temb[2])
        t[5] = float("nan")
        temb, rows = _spread(kernels.time_tokens(emb, proj, t, 256, 10000, 1.0, BF16))
        assert bool(temb[5].isnan().all()) and bool(rows[5].isnan().all()) and int(temb.isnan().any(1).sum()) == 1 and int(rows.isnan().any(1).sum()) == 1


def test_refused(gpu):
    emb, proj = _modules(gpu, BF16, 1536, 9216)
    t = torch.zeros(2706, device=gpu)
    assert kernels.time_tokens(emb, proj, t, 256, 10000, 1.0, BF16) is None  # with gradients
    with torch.inference_mode():
        assert kernels.time_tokens(emb, proj, t, 256, 10000, 1.0, BF16) is not None
        assert kernels.time_tokens(emb, proj, t[:40], 256, 10000, 1.0, BF16) is None  # not for the tile kernel
        assert kernels.time_tokens(emb, proj, t, 256, 10000, 1.0, F16) is None
        assert kernels.time_tokens(emb, proj, t, 128, 10000, 1.0, BF16) is None
        proj.register_forward_hook(lambda *a: None)
        assert kernels.time_tokens(emb, proj, t, 256, 10000, 1.0, BF16) is None
    lib, a = _lib.load(), _lib.TimeTokens()
    assert lib.odit_time_tokens(_lib.C.addressof(a), None, 0, _lib.ODIT_F32, _lib.ODIT_BF16, None, 0, None) == -1
    assert lib.odit_time_tokens_bytes(0, 256, 1536) == 0


def test_captured(gpu):
    """Which way the rows come is found when the graph runs."""
    emb, proj = _modules(gpu, BF16, 1536, 9216)
    t = torch.zeros(2706, device=gpu)
    with torch.inference_mode():
        kernels.time_tokens(emb, proj, t, 256, 10000, 1.0, BF16)
        graph, stream = torch.cuda.CUDAGraph(), torch.cuda.Stream()
        with torch.cuda.graph(graph, stream=stream):
            out = kernels.time_tokens(emb, proj, t, 256, 10000, 1.0, BF16)
        for distinct in (1, 3, 700, 2, 5):
            t.copy_(torch.arange(2706, device=gpu) % distinct)
            graph.replay()
            want = _spread(kernels.time_tokens(emb, proj, t, 256, 10000, 1.0, BF16))
            assert all(torch.equal(a, b) for a, b in zip(_spread(out), want, strict=True))


# widths of every number of wavefronts to a row, and one that takes the general kernel
@pytest.mark.parametrize("S,C", [(1, 512), (77, 1024), (300, 1536), (5, 3072), (129, 4096), (33, 5120), (64, 6152), (9, 8192)])
@pytest.mark.parametrize("dtype", [BF16, F16])
def test_rows_by_number(gpu, S, C, dtype):
    """A table's rows by number give the bits of the same rows written out for every token."""
    print(f"rows by number {S} x {C} {dtype}", flush=True)
    g = torch.Generator(device=gpu).manual_seed(S)
    rand = lambda *s: torch.randn(*s, device=gpu, generator=g)  # noqa: E731
    x, y, table, rows = rand(1, S, C).to(dtype), rand(1, S, C).to(dtype), rand(6, C), rand(7, 6, C).to(dtype)
    rows[5] = float("nan")  # (of no token)
    index = torch.randint(5, (S,), device=gpu, generator=g, dtype=torch.int32)
    full = rows.index_select(0, index).unsqueeze(0)
    with torch.inference_mode():
        got = kernels.adaln_rows(x, rows[:, 0], rows[:, 1], index, table[0], table[1], 1e-6)
        assert torch.equal(got, kernels.adaln_modulate(x, full[:, :, 0], full[:, :, 1], eps=1e-6, shift_bias=table[0], scale_bias=table[1]))
        lib, ptr = _lib.load(), lambda t: None if t is None else t.data_ptr()  # noqa: E731
        for norm in (True, False):
            out, n = torch.full_like(x, -1), torch.full_like(x, -1) if norm else None
            lw, lb = (rand(C), rand(C)) if norm else (None, None)
            gate = rows[:, 2]
            rc = lib.odit_gated_residual_adaln_rows(ptr(x), ptr(y), ptr(gate), ptr(table[2]), ptr(out), ptr(lw), ptr(lb), ptr(n), ptr(index), S, C, 6 * C, 1e-6,
                                                    _lib.ODIT_BF16 if dtype == BF16 else _lib.ODIT_F16, torch.cuda.current_stream().cuda_stream)
            assert rc == 0 and torch.equal(out, kernels.gated_residual(x, y, full[:, :, 2], gate_bias=table[2]))
            if norm:  # a LayerNorm of the rounded row: one rounding of the result, the kernels' float32 sums
                want = torch.nn.functional.layer_norm(out.double(), (C,), lw.double(), lb.double(), 1e-6)
                assert float(((n.double() - want).abs() / (1 + want.abs())).max()) < (2.0 ** -8 if dtype == BF16 else 2.0 ** -10)


def test_model(gpu, monkeypatch):
    """A model with a timestep per token: rows by number where blocks and head are the plain ones, written out where a hook looks on."""
    from vllm_omni_amd.blocks.wan import TokenRows, WanTransformer3DModel

    g = torch.Generator(device=gpu).manual_seed(3)
    model = WanTransformer3DModel(num_attention_heads=12, attention_head_dim=128, ffn_dim=2048, num_layers=2, text_dim=256, cross_attn_norm=True).to(device=gpu, dtype=BF16)
    with torch.no_grad():
        for p in model.parameters():
            p.normal_(0.0, 0.03, generator=g)
    x, text = torch.randn(1, 16, 5, 40, 48, device=gpu, generator=g).to(BF16), torch.randn(1, 20, 256, device=gpu, generator=g).to(BF16)
    t = torch.full((1, 5, 480), 700.0, device=gpu)
    t[:, 0] = 0
    made = []
    full = TokenRows.full
    monkeypatch.setattr(TokenRows, "full", lambda self: made.append(1) or full(self))
    with torch.inference_mode():
        got = model(x, t.flatten(1), text, return_dict=False)[0]
        assert not made
        seen = []
        handle = model.blocks[1].register_forward_pre_hook(lambda m, a: seen.append(a[2].shape))
        again = model(x, t.flatten(1), text, return_dict=False)[0]
        handle.remove()
        assert seen == [(1, 2400, 6, 1536)] and len(made) == 1 and bool(torch.isfinite(got).all())
        monkeypatch.setattr(kernels, "time_tokens", lambda *a: None)
        before = model(x, t.flatten(1), text, return_dict=False)[0]
    scale = float(before.float().norm())
    # the same rows but for last bits of float32 sums: far less than the type's own rounding, half a step in every element
    assert float((got.float() - again.float()).norm()) < 2.0 ** -8 * scale and float((got.float() - before.float()).norm()) < 2.0 ** -8 * scale


@pytest.mark.parametrize("n", [1025, 8192, 8193, 20000])
@pytest.mark.parametrize("places", [(0, 63), (64, 1023), (1024, 65), (8191, 8192), (8192, 16384, 19998), (1, 2, 1025, 9000), (1, 2, 3, 1024), (5, 700, 1000, 1024, 8200)])
def test_where_a_timestep_stands_first(gpu, n, places):
    """One token of its kind at the borders of the search's wavefronts and trips: numbers by timestep, whichever comes first."""
    print(f"timesteps of {n} tokens, alone at {places}", flush=True)
    emb, proj = _modules(gpu, BF16, 512, 3072)
    t = torch.full((n,), 500.0, device=gpu)
    t[n - 1] = 1.0
    for j, at in enumerate(places):
        if at < n:
            t[at] = 600.0 + j
    with torch.inference_mode():
        index = kernels.time_tokens(emb, proj, t, 256, 10000, 1.0, BF16)[2].long()
    values = t.unique()
    if len(values) > 4:
        assert torch.equal(index, torch.arange(n, device=gpu))
    else:
        numbers = [index[t == v].unique() for v in values]
        assert all(len(i) == 1 for i in numbers) and sorted(int(i) for i in numbers) == list(range(len(values)))


@pytest.mark.parametrize("distinct", [2, 5])
def test_two_videos(gpu, distinct):
    """A batch goes the way it always went, whatever its timesteps: each video's result is that of the video alone but for the order of float32 sums."""
    from vllm_omni_amd.blocks.wan import WanTransformer3DModel

    g = torch.Generator(device=gpu).manual_seed(7)
    model = WanTransformer3DModel(num_attention_heads=12, attention_head_dim=128, ffn_dim=2048, num_layers=2, text_dim=256, cross_attn_norm=True).to(device=gpu, dtype=BF16)
    with torch.no_grad():
        for p in model.parameters():
            p.normal_(0.0, 0.03, generator=g)
    x, text = torch.randn(2, 16, 5, 40, 48, device=gpu, generator=g).to(BF16), torch.randn(2, 20, 256, device=gpu, generator=g).to(BF16)
    t = (torch.arange(2400, device=gpu) % distinct * 200.0)[None] + torch.tensor([[0.0], [37.0]], device=gpu)
    with torch.inference_mode():
        both = model(x, t, text, return_dict=False)[0]
        for i in range(2):
            one = model(x[i:i + 1], t[i:i + 1], text[i:i + 1], return_dict=False)[0][0]
            # (last bits of float32 sums: far less than the type's own rounding, half a step in every element)
            assert bool(torch.isfinite(one).all()) and float((both[i].float() - one.float()).norm()) < 2.0 ** -8 * float(one.float().norm())


@pytest.mark.parametrize("distinct", [2, 5])
@pytest.mark.parametrize("dtype", [BF16, F16])
def test_first_product_by_another_kernel(gpu, dtype, distinct):
    """96 cosines and sines: a reduction that the tile kernel does not take, so the first product of all tokens is made in either case."""
    print(f"96 sinusoids, {distinct} distinct {dtype}", flush=True)
    torch.manual_seed(distinct)
    emb, proj = TimestepEmbedding(96, 1536).to(device=gpu, dtype=dtype), torch.nn.Linear(1536, 9216, device=gpu, dtype=dtype)
    t = torch.arange(2706, device=gpu) % distinct * 100.0
    with torch.inference_mode(), torch.profiler.profile(activities=[torch.profiler.ProfilerActivity.CUDA]) as prof:
        got = _spread(kernels.time_tokens(emb, proj, t, 96, 10000, 1.0, dtype))
        torch.cuda.synchronize()
    assert any("token_sinusoid_kernel" in e.key for e in prof.key_averages())
    with torch.inference_mode():
        temb = emb(QwenTimestepProjEmbeddings.time_proj(t, dim=96, scale=1.0, dtype=dtype))
        # the same sums in another order and their roundings, three products deep
        for a, b in zip(got, (temb, kernels.project(proj, temb, silu_input=True)), strict=True):
            assert bool(torch.isfinite(a).all()) and float((a.double() - b.double()).norm()) < (2.0 ** -7 if dtype == BF16 else 2.0 ** -10) * float(b.double().norm())
