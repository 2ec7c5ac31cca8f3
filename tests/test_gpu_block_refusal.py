"""What a kernel inside a native block refuses goes to the Python block instead of failing the forward."""

import pytest
import torch

from test_gpu_native_path import _flux, _init, _qwen, _wan
from vllm_omni_amd import kernels

pytestmark = pytest.mark.gpu


def test_refused_workspace_leaves_the_block_to_python(gpu, monkeypatch):
    from vllm_omni_amd.blocks.qwen_image import QwenImageTransformer2DModel

    model = _init(QwenImageTransformer2DModel(num_layers=1, attention_head_dim=64, num_attention_heads=4, joint_attention_dim=256,
                                              axes_dims_rope=(8, 28, 28)), gpu, torch.bfloat16)
    model.fuse_modulation()
    # 66 query blocks of 128 rows x 8 (batch, head) pairs: a few more than run at once, whose keys are split through scratch
    lat, enc = torch.randn(2, 128 * 65 + 64, 64, device=gpu).bfloat16(), torch.randn(2, 64, 256, device=gpu).bfloat16()
    t = torch.full((2,), 0.3, device=gpu).bfloat16()
    assert ";" in kernels.attn_plan(2, 128 * 66, 128 * 66, 4, 64)
    nat, asked = kernels.native(), []

    def too_small(device, stream, need):
        asked.append(need)
        return kernels._attn_scratch(device, stream, need) if len(asked) > 1 else torch.zeros(16, dtype=torch.uint8, device=gpu)

    side = torch.cuda.Stream()   # (no scratch known for it yet)
    torch.cuda.synchronize()
    with torch.inference_mode(), torch.cuda.stream(side):
        call = lambda: model(lat, enc, None, t, [(1, 64, 131)], [64, 64]).sample  # noqa: E731
        nat.configure(kernels._linear_scratch, too_small)
        try:
            got = call()
        finally:
            nat.configure(kernels._linear_scratch, kernels._attn_scratch)
        monkeypatch.setattr(kernels, "NATIVE_BLOCKS", False)
        want = call()
    side.synchronize()
    assert len(asked) >= 2 and torch.equal(got, want)


def _off_by_one(p):
    """The same values at an address that is 2 bytes past a 16-byte boundary."""
    buf = torch.empty(p.numel() + 8, dtype=p.dtype, device=p.device)
    view = buf[1:p.numel() + 1].view(p.shape)
    view.copy_(p)
    return torch.nn.Parameter(view, requires_grad=False)


@pytest.mark.parametrize("which", ["weight", "bias"])
def test_misaligned_parameters_are_left_to_torch(gpu, which):
    """Nothing is launched: the answers say so."""
    lin = torch.nn.Linear(256, 192, device=gpu, dtype=torch.bfloat16)
    x = torch.randn(40, 256, device=gpu).bfloat16()
    with torch.inference_mode():
        assert kernels.native().project(lin, x, False, 0) is not None
        assert kernels.native().project(lin, torch.cat([x, x]).flatten()[1:40 * 256 + 1].view(40, 256), False, 0) is None
        setattr(lin, which, _off_by_one(getattr(lin, which).detach()))
        assert kernels.native().project(lin, x, False, 0) is None


@pytest.mark.parametrize("make,name,pick", [(_qwen, "qwen_block", lambda m: m.transformer_blocks[-1].attn.to_qkv),
                                            (_flux, "flux_single_block", lambda m: m.single_transformer_blocks[-1].proj_mlp),
                                            (_wan, "wan_block", lambda m: m.blocks[-1].attn2.to_k)])
def test_blocks_with_a_misaligned_weight_are_left_to_python(gpu, make, name, pick):
    model, call = make(gpu, torch.bfloat16, 64, False)
    nat, args = kernels.native(), []

    class Recorder:
        def __getattr__(self, n):
            if n != name:
                return getattr(nat, n)
            return lambda *a: (args.append(a), getattr(nat, n)(*a))[1]

    with torch.inference_mode():
        kernels._nat = Recorder()
        try:
            call()
        finally:
            kernels._nat = nat
        assert getattr(nat, name)(*args[-1]) is not None
        lin = pick(model)
        lin.weight = _off_by_one(lin.weight.detach())
        assert getattr(nat, name)(*args[-1]) is None
