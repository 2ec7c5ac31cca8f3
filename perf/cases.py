"""The work that users of this package have it do, as cases that can be timed and compared.

Each case goes through the public classes: the denoise loops around the three transformer families (the
reference's CFG mixin for Qwen-Image, ``diffuse_flux`` with and without TeaCache, the Wan model with its CFG
pair), and the layers that are dropped into an existing install one by one (attention, adaLN, QK norm, rotary).
Widths are those of BASELINE.json's configurations. Every block of a model costs the same, so the models have a
few blocks each; sequence lengths, batch, masks and prompt lengths are what a request brings.
"""

import math

import torch

from vllm_omni_amd import denoise, gemm_tuning
from vllm_omni_amd.attention.backends.abstract import AttentionMetadata
from vllm_omni_amd.attention.layer import Attention
from vllm_omni_amd.blocks.flux import FluxTransformer2DModel
from vllm_omni_amd.blocks.qwen_image import QwenImageTransformer2DModel
from vllm_omni_amd.blocks.wan import WanTransformer3DModel
from vllm_omni_amd.cache.teacache import TeaCacheBackend
from vllm_omni_amd.layers import AdaLayerNorm, RMSNorm, RotaryEmbedding

_DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16}
_DEVICE = "cuda"


# ------------------------------------------------------------------------------------------------ cases
def listed():
    return [
        # a whole 4-step generation with the smallest model: launches and host time
        dict(name="qwen_tiny_4steps", kind="qwen", heads=4, head_dim=64, layers=2, text_dim=256, h=16, w=16, txt=64,
             neg=0, edit_h=0, edit_w=0, steps=4, dtype="bf16"),
        # a thumbnail or preview: 256 x 256 pixels, short prompts; the weights are read for few rows
        dict(name="qwen_256px_preview", kind="qwen", heads=24, head_dim=128, layers=12, text_dim=3584, h=16, w=16, txt=40,
             neg=40, edit_h=0, edit_w=0, steps=1, dtype="bf16"),
        # 512 x 512 with a long prompt against a short negative one: padded and masked in the CFG batch
        dict(name="qwen_512px_two_prompts", kind="qwen", heads=24, head_dim=128, layers=8, text_dim=3584, h=32, w=32,
             txt=171, neg=23, edit_h=0, edit_w=0, steps=1, dtype="bf16"),
        # the headline shape: 1024 x 1024, CFG batch 2, 256 text tokens
        dict(name="qwen_1024px", kind="qwen", heads=24, head_dim=128, layers=6, text_dim=3584, h=64, w=64, txt=256, neg=256,
             edit_h=0, edit_w=0, steps=1, dtype="bf16"),
        # image editing (per-token conditioning): a 16:9 target beside its source image, ragged lengths
        dict(name="qwen_edit_16x9", kind="qwen", heads=24, head_dim=128, layers=4, text_dim=3584, h=36, w=64, txt=203,
             neg=203, edit_h=39, edit_w=59, steps=1, dtype="bf16"),
        # guidance-distilled Flux at 512 x 512: batch 1
        dict(name="flux_512px", kind="flux", dual=4, single=8, h=32, w=32, txt=512, steps=1, teacache=0.0, dtype="bf16"),
        # Flux at 1024 x 1024 under the TeaCache hook: computed and skipped steps, one decision each
        dict(name="flux_1024px_teacache", kind="flux", dual=3, single=6, h=64, w=64, txt=512, steps=8, teacache=0.6,
             dtype="bf16"),
        # text-to-video: 81 frames at 480 x 832 (21 x 30 x 52 = 32760 tokens), CFG batch 2: the largest
        dict(name="wan_480p_81frames", kind="wan", layers=2, frames=21, h=30, w=52, txt=512, batch=2, per_token=False,
             dtype="bf16"),
        # image-to-video conditioning with a timestep per token, a short clip on a ragged grid
        dict(name="wan_per_token_clip", kind="wan", layers=3, frames=3, h=22, w=41, txt=512, batch=1, per_token=True,
             dtype="bf16"),
        # the attention layer alone in an existing model: grouped heads, padded keys, fp16
        dict(name="attention_fp16_padded", kind="attention", batch=2, sq=1357, sk=1357, heads=32, kv_heads=8, head_dim=64,
             masked=True, dtype="fp16"),
        # the norm, modulation and rotary layers alone: the text stream of one prompt
        dict(name="layers_text", kind="layers", batch=1, seq=77, heads=24, head_dim=128, dtype="bf16"),
        # and the image stream of a CFG pair
        dict(name="layers_image", kind="layers", batch=2, seq=6032, heads=24, head_dim=128, dtype="fp16"),
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    while True:
        case = _draw_one(rng)
        if _cost(case) <= _MOST_COST:
            return case


def _draw_one(rng):
    dtype = rng.choice(("bf16", "bf16", "bf16", "fp16"))
    kind = rng.choice(("qwen", "qwen", "qwen", "flux", "flux", "wan", "wan", "attention", "layers"))
    if kind == "qwen":
        tiny = rng.random() < 0.15
        tokens, aspect = _log_int(rng, 128, 7000), math.exp(rng.uniform(-0.6, 0.6))
        h = max(4, round(math.sqrt(tokens * aspect)))
        edit = not tiny and rng.random() < 0.2
        txt = _log_int(rng, 8, 512)
        neg = rng.choice((0, txt, txt, _log_int(rng, 8, 512)))
        return dict(kind="qwen", heads=4 if tiny else 24, head_dim=64 if tiny else 128,
                    layers=2 if tiny else rng.randint(2, 8), text_dim=256 if tiny else 3584, h=h, w=max(4, tokens // h),
                    txt=txt, neg=neg, edit_h=rng.randint(16, 48) if edit else 0, edit_w=rng.randint(16, 48) if edit else 0,
                    steps=rng.randint(1, 4) if tiny else 1, dtype=dtype)
    if kind == "flux":
        tokens, aspect = _log_int(rng, 128, 7000), math.exp(rng.uniform(-0.6, 0.6))
        h = max(4, round(math.sqrt(tokens * aspect)))
        cached = rng.random() < 0.3
        return dict(kind="flux", dual=rng.randint(1, 3), single=rng.randint(2, 6), h=h, w=max(4, tokens // h),
                    txt=rng.choice((256, 512, _log_int(rng, 16, 512))), steps=8 if cached else 1,
                    teacache=0.6 if cached else 0.0, dtype=dtype)
    if kind == "wan":
        frames, h = rng.randint(1, 21), rng.randint(8, 45)
        return dict(kind="wan", layers=rng.randint(1, 3), frames=frames, h=h, w=rng.randint(8, 80),
                    txt=rng.choice((512, 512, _log_int(rng, 16, 512))), batch=rng.randint(1, 2), per_token=rng.random() < 0.3,
                    dtype=dtype)
    if kind == "attention":
        heads = rng.choice((8, 16, 24, 32, 40))
        sq = _log_int(rng, 16, 16384)
        return dict(kind="attention", batch=rng.randint(1, 4), sq=sq, sk=sq if rng.random() < 0.6 else _log_int(rng, 16, 1024),
                    heads=heads, kv_heads=heads // rng.choice((1, 1, 4)), head_dim=rng.choice((64, 128)),
                    masked=rng.random() < 0.4, dtype=dtype)
    heads = rng.choice((8, 12, 24, 40))
    return dict(kind="layers", batch=rng.randint(1, 2), seq=_log_int(rng, 16, 16384), heads=heads,
                head_dim=rng.choice((64, 128)), dtype=dtype)


# --------------------------------------------------------------------------------------------- prepare
def _generator(seed):
    return torch.Generator(device=_DEVICE).manual_seed(seed)


def _randn(g, dtype, *shape):
    return torch.randn(*shape, device=_DEVICE, generator=g).to(dtype)


def _built(make, dtype, g):
    """A model on the GPU with synthetic weights: N(0, 0.02) matrices and biases, norm weights about one."""
    prev = torch.get_default_dtype()
    torch.set_default_dtype(dtype)
    try:
        with torch.device(_DEVICE):
            model = make()
    finally:
        torch.set_default_dtype(prev)
    with torch.no_grad():
        for name, p in model.named_parameters():
            if name.endswith("scale_shift_table"):
                p.normal_(0.0, p.shape[-1] ** -0.5, generator=g)
            elif "norm" in name and name.endswith(".weight") and p.dim() == 1:
                p.normal_(1.0, 0.1, generator=g)
            else:
                p.normal_(0.0, 0.02, generator=g)
    if hasattr(model, "fuse_modulation"):
        model.fuse_modulation()
    return model.eval()


class _QwenPipeline(denoise.QwenImageCFGParallelMixin):
    def __init__(self, transformer):
        self.transformer, self.scheduler = transformer, denoise.FlowMatchEulerScheduler()


class _FluxPipeline:
    def __init__(self, transformer):
        self.transformer = transformer


def _prepare_qwen(c, g, dtype):
    edit = c["edit_h"] > 0
    axes = (16, 56, 56) if c["head_dim"] == 128 else (8, 28, 28)
    model = _built(lambda: QwenImageTransformer2DModel(
        num_layers=c["layers"], attention_head_dim=c["head_dim"], num_attention_heads=c["heads"],
        joint_attention_dim=c["text_dim"], axes_dims_rope=axes, zero_cond_t=edit), dtype, g)
    pipe, tokens = _QwenPipeline(model), c["h"] * c["w"]
    pipe.scheduler.set_timesteps(max(c["steps"], 20), device=_DEVICE, mu=denoise.calculate_shift(tokens))
    shapes = [(1, c["h"], c["w"])] + ([(1, c["edit_h"], c["edit_w"])] if edit else [])
    neg = c["neg"] > 0
    args = dict(
        prompt_embeds=_randn(g, dtype, 1, c["txt"], c["text_dim"]), prompt_embeds_mask=None,
        negative_prompt_embeds=_randn(g, dtype, 1, c["neg"], c["text_dim"]) if neg else None,
        negative_prompt_embeds_mask=None, latents=_randn(g, dtype, 1, tokens, 64), img_shapes=[shapes],
        txt_seq_lens=[c["txt"]], negative_txt_seq_lens=[c["neg"]] if neg else None,
        timesteps=pipe.scheduler.timesteps[:c["steps"]], do_true_cfg=neg, guidance=None, true_cfg_scale=4.0,
        image_latents=_randn(g, dtype, 1, c["edit_h"] * c["edit_w"], 64) if edit else None)
    return dict(pipe=pipe, args=args)


def _prepare_flux(c, g, dtype):
    model = _built(lambda: FluxTransformer2DModel(num_layers=c["dual"], num_single_layers=c["single"]), dtype, g)
    pipe, cache = _FluxPipeline(model), None
    if c["teacache"] > 0:
        cache = TeaCacheBackend({"rel_l1_thresh": c["teacache"]})
        cache.enable(pipe)
    ids = torch.zeros(c["h"], c["w"], 3, device=_DEVICE)
    ids[..., 1] += torch.arange(c["h"], device=_DEVICE)[:, None]
    ids[..., 2] += torch.arange(c["w"], device=_DEVICE)[None, :]
    args = dict(latents=_randn(g, dtype, 1, c["h"] * c["w"], 64), prompt_embeds=_randn(g, dtype, 1, c["txt"], 4096),
                pooled_prompt_embeds=_randn(g, dtype, 1, 768), img_ids=ids.reshape(-1, 3),
                txt_ids=torch.zeros(c["txt"], 3, device=_DEVICE), num_inference_steps=c["steps"])
    return dict(pipe=pipe, cache=cache, args=args, steps=c["steps"])


def _prepare_wan(c, g, dtype):
    model = _built(lambda: WanTransformer3DModel(num_layers=c["layers"]), dtype, g)
    frames, h, w = c["frames"], c["h"], c["w"]
    if c["per_token"]:  # the first frame is given (timestep zero), the others are denoised
        t = torch.full((c["batch"], frames, h * w), 700.0, device=_DEVICE)
        t[:, 0] = 0.0
        t = t.flatten(1)
    else:
        t = torch.full((c["batch"],), 700.0, device=_DEVICE)
    return dict(model=model, latents=_randn(g, dtype, 1, 16, frames, 2 * h, 2 * w), timestep=t, batch=c["batch"],
                text=_randn(g, dtype, c["batch"], c["txt"], 4096))


def _prepare_attention(c, g, dtype):
    layer = Attention(num_heads=c["heads"], head_size=c["head_dim"], causal=False, softmax_scale=c["head_dim"] ** -0.5,
                      num_kv_heads=c["kv_heads"])
    q = _randn(g, dtype, c["batch"], c["sq"], c["heads"], c["head_dim"])
    k = _randn(g, dtype, c["batch"], c["sk"], c["kv_heads"], c["head_dim"])
    v = _randn(g, dtype, c["batch"], c["sk"], c["kv_heads"], c["head_dim"])
    meta = None
    if c["masked"]:  # sequences of unequal length, padded to the longest
        lens = torch.randint(max(1, c["sk"] // 3), c["sk"] + 1, (c["batch"],), device=_DEVICE, generator=g)
        lens[0] = c["sk"]
        meta = AttentionMetadata(attn_mask=torch.arange(c["sk"], device=_DEVICE)[None, :] < lens[:, None])
    return dict(layer=layer, q=q, k=k, v=v, meta=meta)


def _prepare_layers(c, g, dtype):
    width = c["heads"] * c["head_dim"]
    norms = _built(lambda: torch.nn.ModuleDict(dict(norm_q=RMSNorm(c["head_dim"]), norm_k=RMSNorm(c["head_dim"]))), dtype, g)
    angles = torch.rand(c["seq"], c["head_dim"] // 2, device=_DEVICE, generator=g) * 6.2831853
    return dict(adaln=AdaLayerNorm(width), norms=norms, rope=RotaryEmbedding(), cos=angles.cos(), sin=angles.sin(),
                x=_randn(g, dtype, c["batch"], c["seq"], width), mod=_randn(g, dtype, c["batch"], 3 * width),
                q=_randn(g, dtype, c["batch"], c["seq"], c["heads"], c["head_dim"]),
                k=_randn(g, dtype, c["batch"], c["seq"], c["heads"], c["head_dim"]))


_PREPARE = {"qwen": _prepare_qwen, "flux": _prepare_flux, "wan": _prepare_wan, "attention": _prepare_attention,
            "layers": _prepare_layers}
_tuned = []


def prepare(case, seed):
    if not _tuned:  # once per process, as a program does at start-up
        _tuned.append(gemm_tuning.enable())
    with torch.no_grad():
        state = _PREPARE[case["kind"]](case, _generator(seed), _DTYPES[case["dtype"]])
    state["kind"] = case["kind"]
    return state


# ------------------------------------------------------------------------------------------------- run
def _run_qwen(s):
    return s["pipe"].diffuse(**s["args"])


def _run_flux(s):
    if s["cache"] is not None:
        s["cache"].refresh(s["pipe"], s["steps"])
    return denoise.diffuse_flux(s["pipe"].transformer, **s["args"])


def _run_wan(s):
    x = s["latents"].expand(s["batch"], -1, -1, -1, -1)
    noise = s["model"](x, s["timestep"], s["text"], return_dict=False)[0]
    if s["batch"] == 2:
        noise = denoise.combine_cfg_noise(noise[0:1], noise[1:2], 5.0, False)
    return [noise, denoise.euler_step(s["latents"], noise, 0.70, 0.66)]


def _run_attention(s):
    return s["layer"](s["q"], s["k"], s["v"], s["meta"])


def _run_layers(s):
    out, gate = s["adaln"](s["x"], s["mod"])
    q = s["rope"](s["norms"]["norm_q"](s["q"]), s["cos"], s["sin"])
    k = s["rope"](s["norms"]["norm_k"](s["k"]), s["cos"], s["sin"])
    return [out, gate, q, k]


_RUN = {"qwen": _run_qwen, "flux": _run_flux, "wan": _run_wan, "attention": _run_attention, "layers": _run_layers}


def run(state):
    with torch.inference_mode():
        return _RUN[state["kind"]](state)


# ------------------------------------------------------------------------------------------------ work
def _qwen_work(c):
    C, L, B = c["heads"] * c["head_dim"], c["layers"], 2 if c["neg"] else 1
    img, txt = c["h"] * c["w"] + c["edit_h"] * c["edit_w"], max(c["txt"], c["neg"])
    rows = c["txt"] + c["neg"] + B * img
    block = 12 * C * C  # per stream: qkv 3, out 1, MLP 8
    weights = L * (2 * block + 12 * C * C) + C * (64 + c["text_dim"] + 256 + C) + C * (2 * C + 64)
    cond = 2 * B if c["edit_h"] else B
    flops = L * (2 * rows * block + 2 * (cond + B) * 6 * C * C)
    for t in ([c["txt"], c["neg"]] if c["neg"] else [txt]):
        flops += L * 4 * (t + img) ** 2 * C
    io = 2 * (c["txt"] + c["neg"]) * c["text_dim"] + 2 * (c["h"] * c["w"] * 2 + c["edit_h"] * c["edit_w"]) * 64
    return c["steps"] * (2 * weights + io), c["steps"] * flops


def _flux_work(c):
    C, S = 3072, c["h"] * c["w"] + c["txt"]
    weights = c["dual"] * (24 + 12) * C * C + c["single"] * (12 + 3) * C * C + C * (64 + 4096 + 2 * 256 + 768 + 5 * C + 64)
    flops = (c["dual"] + c["single"]) * (2 * S * 12 * C * C + 4 * S * S * C)
    steps = c["steps"]
    full = steps if c["teacache"] == 0 else (3 * steps + 7) // 8  # 0.6 computes 3 steps of 8
    io = 2 * c["h"] * c["w"] * 64 * 2 + 2 * c["txt"] * 4096
    return full * 2 * weights + steps * io, full * flops


def _wan_work(c):
    C, F, B, S = 5120, 13824, c["batch"], c["frames"] * c["h"] * c["w"]
    weights = c["layers"] * (8 * C * C + 2 * C * F) + C * (64 + 256 + C + 6 * C + 4096 + C + 64)
    flops = c["layers"] * B * (2 * S * (6 * C * C + 2 * C * F) + 2 * c["txt"] * 2 * C * C + 4 * S * (S + c["txt"]) * C)
    if c["per_token"]:
        flops += 2 * B * S * C * (256 + 7 * C)
    io = 2 * (B * S * 64 + 2 * S * 64 + B * c["txt"] * 4096)
    return 2 * weights + io, flops


def _attention_work(c):
    q = c["batch"] * c["sq"] * c["heads"] * c["head_dim"]
    kv = c["batch"] * c["sk"] * c["kv_heads"] * c["head_dim"]
    keys = 0.75 if c["masked"] else 1.0  # mean length of the padded sequences
    return 2 * (2 * q + 2 * kv), keys * 4 * q * c["sk"]


def _layers_work(c):
    n = c["batch"] * c["seq"] * c["heads"] * c["head_dim"]
    return 2 * 6 * n + 4 * c["seq"] * c["head_dim"], 30 * n


_WORK = {"qwen": _qwen_work, "flux": _flux_work, "wan": _wan_work, "attention": _attention_work, "layers": _layers_work}


def work(case):
    nbytes, flops = _WORK[case["kind"]](case)
    return {"bytes": nbytes, "flops": flops}


def _cost(case):
    nbytes, flops = _WORK[case["kind"]](case)
    return max(flops, 200 * nbytes)


_MOST_COST = max(_cost(c) for c in listed())


def tolerance(case):
    # 16-bit activations are rounded at every operation of every block; the layers alone round once or twice
    if case["kind"] in ("attention", "layers"):
        return {"rel": 1e-2 if case["dtype"] == "bf16" else 2e-3}
    return {"rel": 1.5e-2 if case["dtype"] == "bf16" else 4e-3}
