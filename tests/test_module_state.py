"""What the models form from their parameters follows the parameters, however they are written (CPU)."""

import pytest
import torch


def _write(p, value, how):
    if how == "data":        # the usual form of a weight loader: neither the version counter nor the address changes
        p.data.copy_(value)
    else:
        with torch.no_grad():
            p.copy_(value)


def _random_(model):
    g = torch.Generator().manual_seed(0)
    for p in model.parameters():
        p.data.copy_(torch.randn(p.shape, generator=g) * 0.1)
    return model


@pytest.mark.parametrize("how", ["data", "in place"])
def test_qwen_gate_rows_follow_the_biases(how):
    from vllm_omni_amd.blocks.qwen_image import QwenImageTransformer2DModel

    model = _random_(QwenImageTransformer2DModel(num_layers=2, attention_head_dim=64, num_attention_heads=1, joint_attention_dim=64,
                                                 axes_dims_rope=(8, 28, 28)).to(torch.bfloat16))
    mods = torch.randn(2, 2, 2, 6 * 64).to(torch.bfloat16)
    model.all_gate_rows(mods)
    for i, pick in enumerate((lambda b: b.attn.to_out, lambda b: b.img_mlp.net[2], lambda b: b.attn.to_add_out, lambda b: b.txt_mlp.net[2])):
        bias = pick(model.transformer_blocks[1]).bias
        _write(bias, torch.full_like(bias, 0.5 + i), how)
        gates, gb = model.all_gate_rows(mods)
        assert gb.dtype == torch.float32
        assert torch.equal(gb[:, 1, i // 2, i % 2], gates[:, 1, i // 2, i % 2] * (0.5 + i))


@pytest.mark.parametrize("how", ["data", "in place"])
def test_flux_gate_rows_follow_the_biases(how):
    from vllm_omni_amd.blocks.flux import FluxTransformer2DModel

    model = _random_(FluxTransformer2DModel(num_layers=1, num_single_layers=2, attention_head_dim=64, num_attention_heads=1,
                                            joint_attention_dim=64, pooled_projection_dim=8, axes_dims_rope=(8, 28, 28)).to(torch.bfloat16))
    mods = (torch.randn(2, 1, 2, 6 * 64).to(torch.bfloat16), torch.randn(2, 2, 3 * 64).to(torch.bfloat16))
    model.all_gate_rows(mods)
    dual, single = model.transformer_blocks[0].ff_context.net[2].bias, model.single_transformer_blocks[1].proj_out.bias
    _write(dual, torch.full_like(dual, 0.5), how)
    _write(single, torch.full_like(single, 2.0), how)
    (dg, dgb), (sg, sgb) = model.all_gate_rows(mods)
    assert dgb.dtype == sgb.dtype == torch.float32
    assert torch.equal(dgb[:, 0, 1, 1], dg[:, 0, 1, 1] * 0.5)
    assert torch.equal(sgb[:, 1], sg[:, 1] * 2.0)


@pytest.mark.parametrize("how", ["data", "in place"])
def test_wan_rows_follow_the_parameters(how):
    from vllm_omni_amd.blocks.wan import WanTransformer3DModel

    model = _random_(WanTransformer3DModel(num_attention_heads=1, attention_head_dim=64, text_dim=32, ffn_dim=128, num_layers=2).to(torch.bfloat16))
    mods = torch.randn(2, 3, 6, 64)
    block = model.blocks[1]
    for _ in range(2):  # the second time round whatever the first could have kept is there
        for p in (block.attn1.to_out.bias, block.ffn.net_2.bias, block.norm2.weight, block.norm2.bias, block.scale_shift_table):
            _write(p, torch.randn(p.shape).to(p.dtype), how)
        gb = model.gate_bias_rows(mods)
        # (rows of the gates and of gate * bias have to lie equally far apart from batch entry to batch entry)
        assert gb.shape == (2, 3, 2, 64) and gb.dtype == torch.float32 and gb[1].stride(0) == mods[1].stride(0)
        assert torch.equal(gb[1, :, 0], mods[1, :, 2] * block.attn1.to_out.bias.float())
        assert torch.equal(gb[1, :, 1], mods[1, :, 5] * block.ffn.net_2.bias.float())
        one = (mods[1] * block.gated_biases())[:, 2::3]
        assert torch.equal(one, gb[1])
        for w, b in (model.norm2_affines()[1], block._norm2_affine()):
            assert torch.equal(w, block.norm2.weight.float()) and torch.equal(b, block.norm2.bias.float())
        assert torch.equal(block._table(), block.scale_shift_table[0].float())


def _qwen_stem():
    from vllm_omni_amd.blocks.qwen_image import QwenImageTransformer2DModel

    model = QwenImageTransformer2DModel(num_layers=1, attention_head_dim=64, num_attention_heads=1, joint_attention_dim=64,
                                        axes_dims_rope=(8, 28, 28))
    return model, model.transformer_blocks[0].img_mod[1], (None, None, None, None, None, None)


def _flux_stem():
    from vllm_omni_amd.blocks.flux import FluxTransformer2DModel

    model = FluxTransformer2DModel(num_layers=1, num_single_layers=0, attention_head_dim=64, num_attention_heads=1,
                                   joint_attention_dim=64, pooled_projection_dim=8, axes_dims_rope=(8, 28, 28))
    return model, model.transformer_blocks[0].norm1.linear, (None,) * 6


def _decision_rows(monkeypatch, model, args):
    """The shift and scale that the cache decision is made with, on a given stem output."""
    from vllm_omni_amd import kernels
    from vllm_omni_amd.cache.teacache.extractors import get_extractor

    img, temb = torch.zeros(2, 3, 64), torch.linspace(-1, 1, 128).view(2, 64)
    monkeypatch.setattr(model, "prepare", lambda *a, **k: (img, None, temb, None), raising=False)
    monkeypatch.setattr(kernels, "silu", torch.nn.functional.silu)
    rows = []
    monkeypatch.setattr(kernels, "adaln_modulate", lambda x, shift, scale, **k: rows.extend((shift, scale)) or x)
    with torch.no_grad():
        get_extractor(type(model).__name__)(model, *args)
    return torch.cat(rows, dim=-1)


@pytest.mark.parametrize("make,how", [(m, h) for m in (_qwen_stem, _flux_stem) for h in ("plain", "hook", "global hook", "own forward")]
                         + [(_qwen_stem, "activation hook")])
def test_cache_decision_projection_is_called_unless_plain(monkeypatch, make, how):
    model, lin, args = make()
    _random_(model)
    want = lin(torch.nn.functional.silu(torch.linspace(-1, 1, 128).view(2, 64)))[:, :128].detach()
    seen, handle = [], None
    if how == "hook":
        lin.register_forward_hook(lambda *a: seen.append(1))
    elif how == "global hook":
        handle = torch.nn.modules.module.register_module_forward_hook(lambda m, *a: seen.append(1) if m is lin else None)
    elif how == "own forward":   # as an offloading wrapper puts it there: the weight is elsewhere between calls
        weight, inner = lin.weight.data, lin.forward

        def forward(x):
            seen.append(1)
            lin.weight.data = weight
            return inner(x)

        lin.forward = forward
        lin.weight.data = torch.empty(0, 64)
    elif how == "activation hook":
        model.transformer_blocks[0].img_mod[0].register_forward_hook(lambda *a: seen.append(1))
    try:
        got = _decision_rows(monkeypatch, model, args)
    finally:
        if handle is not None:
            handle.remove()
    assert seen == ([] if how == "plain" else [1])
    torch.testing.assert_close(got, want)


@pytest.mark.parametrize("batch", [1, 2])
@pytest.mark.parametrize("how", ["hook", "own forward", "replaced"])
def test_wan_time_embedder_is_called(monkeypatch, how, batch):
    from vllm_omni_amd import kernels
    from vllm_omni_amd.blocks.wan import WanTimeTextImageEmbedding

    monkeypatch.setattr(kernels, "silu", torch.nn.functional.silu)
    monkeypatch.setattr(kernels, "gelu_tanh", lambda x, out=None: torch.nn.functional.gelu(x, approximate="tanh"))
    emb = _random_(WanTimeTextImageEmbedding(64, 16, 6 * 64, 32))
    t, text = torch.full((batch,), 500.0), torch.randn(batch, 3, 32)
    seen = []
    with torch.no_grad():
        plain = emb(t, text)
        if how == "hook":
            emb.time_embedder.register_forward_hook(lambda m, a, out: seen.append(1) or 2 * out)
        elif how == "own forward":
            inner = emb.time_embedder.forward
            emb.time_embedder.forward = lambda x: seen.append(1) or 2 * inner(x)
        else:
            class Twice(torch.nn.Module):
                def __init__(self, mlp):
                    super().__init__()
                    self.linear_1, self.linear_2 = mlp.linear_1, mlp.linear_2

                def forward(self, x):
                    seen.append(1)
                    return 2 * self.linear_2(torch.nn.functional.silu(self.linear_1(x)))

            emb.time_embedder = Twice(emb.time_embedder)
        changed = emb(t, text)
    assert seen == [1]
    torch.testing.assert_close(changed[0], 2 * plain[0])


@pytest.mark.parametrize("where", ["class", "instance"])
def test_a_pipelines_own_cfg_normalisation_is_used(where):
    from vllm_omni_amd.denoise import CFGParallelMixin

    class Pipe(CFGParallelMixin):
        pass

    pipe = Pipe()
    if where == "class":
        Pipe.cfg_normalize_function = lambda self, pred, comb: comb * 0 + 7
    else:
        pipe.cfg_normalize_function = lambda pred, comb: comb * 0 + 7
    pos, neg = torch.randn(1, 3, 8), torch.randn(1, 3, 8)
    assert torch.equal(pipe.combine_cfg_noise(pos, neg, 4.0, True), torch.full((1, 3, 8), 7.0))
    torch.testing.assert_close(pipe.combine_cfg_noise(pos, neg, 4.0, False), neg + 4.0 * (pos - neg))


def test_a_replaced_wan_block_gets_the_arguments_it_knows(monkeypatch):
    from vllm_omni_amd.blocks.wan import WanTransformer3DModel

    model = _random_(WanTransformer3DModel(num_attention_heads=1, attention_head_dim=64, text_dim=32, ffn_dim=128, num_layers=2))
    block = model.blocks[0]
    got = []

    def forward(x, ctx, temb, rotary=None, mod=None, gate_bias=None):
        got.append((temb is None, mod is None, gate_bias is None))
        return x + 1

    for b in model.blocks:
        b.forward = forward
    x, ctx = torch.zeros(1, 3, 64), torch.zeros(1, 4, 64)
    assert torch.equal(model.run_blocks(x, ctx, torch.zeros(1, 6, 64), None), x + 2)
    assert torch.equal(model.run_blocks(x, ctx, torch.zeros(1, 3, 6, 64), None), x + 2)
    assert got == [(True, False, True)] * 2 + [(False, True, True)] * 2


@pytest.mark.parametrize("small", [False, True])
def test_qwen_gate_rows_of_somebody_elses(monkeypatch, small):
    """An override with the signature that the method has always had is called in every step, also where this package's would be left out."""
    from vllm_omni_amd import kernels
    from vllm_omni_amd.blocks.qwen_image import QwenImageTransformer2DModel

    seen = []

    class Own(QwenImageTransformer2DModel):
        def all_gate_rows(self, mods):
            seen.append(mods)

    monkeypatch.setattr(kernels, "small_pairs", lambda *a: small)
    monkeypatch.setattr(kernels, "gate_rows", lambda *a: seen.append(a[0]))
    size = dict(num_layers=1, attention_head_dim=64, num_attention_heads=1, joint_attention_dim=64, axes_dims_rope=(8, 28, 28))
    models = [QwenImageTransformer2DModel(**size), Own(**size), QwenImageTransformer2DModel(**size)]
    models[2].all_gate_rows = lambda mods: seen.append(mods)
    mods = torch.zeros(1, 1, 2, 6 * 64, dtype=torch.bfloat16)
    for model, calls in zip(models, (not small, True, True)):
        monkeypatch.setattr(model, "_gated_biases", lambda: [torch.zeros(64)] * 4)
        model.transformer_blocks = torch.nn.ModuleList()
        model.run_blocks(torch.zeros(1, 4, 64), torch.zeros(1, 3, 64), None, None, mods=mods)
        assert len(seen) == calls and all(torch.equal(m, mods) for m in seen)
        seen.clear()


def test_a_qwen_model_saved_whole_earlier(monkeypatch):
    import pickle

    from vllm_omni_amd import kernels
    from vllm_omni_amd.blocks.qwen_image import QwenImageTransformer2DModel

    model = QwenImageTransformer2DModel(num_layers=1, attention_head_dim=64, num_attention_heads=1, joint_attention_dim=64, axes_dims_rope=(8, 28, 28))
    del model._mlp_dim
    model, called = pickle.loads(pickle.dumps(model)), []
    monkeypatch.setattr(kernels, "small_pairs", lambda *a: True)
    monkeypatch.setattr(type(model), "all_gate_rows", lambda self, mods: called.append(mods))
    model.transformer_blocks = torch.nn.ModuleList()
    model.run_blocks(torch.zeros(1, 4, 64), torch.zeros(1, 3, 64), None, None, mods=torch.zeros(1, 1, 2, 6 * 64, dtype=torch.bfloat16))
    assert len(called) == 1
