"""Wan blocks of one video at the model's width, whose text keys and values are projected in the launch of the self-attention's
projection (native.cpp, wan_block): against the same block kernel by kernel. The keys and values then lie in the block's
memory through the self-attention, beside everything else that shares it."""

import pytest
import torch

from test_gpu_native_width import _built, _rand
from vllm_omni_amd import _lib, kernels

pytestmark = pytest.mark.gpu

C = _lib.C
WIDTH = 5120


def _one_launch(rows, text_rows, dtype):
    """What odit_linear_three answers for a block of so many rows."""
    at = torch.zeros(64, device="cuda", dtype=dtype)
    q, widths = (_lib.LinearProblem * 3)(), (3 * WIDTH, WIDTH, WIDTH)
    for i, m in enumerate((rows, text_rows, text_rows)):
        q[i].x = q[i].w = q[i].bias = q[i].out = at.data_ptr()
        q[i].M, q[i].ldx, q[i].ldw, q[i].ldo = m, WIDTH, WIDTH, widths[i]
    stream = torch.cuda.current_stream().cuda_stream
    ws = kernels._linear_scratch(at.device.index or 0, stream)
    return _lib.load().odit_linear_three(C.addressof(q), (C.c_int * 3)(*widths), WIDTH, (C.c_int * 3)(1, 1, 1), 0 if dtype == torch.bfloat16 else 1, 0,
                                         _lib.ODIT_LAUNCH_ASK, ws.data_ptr(), ws.numel(), stream)


# frames, rows and columns of patches, text rows, whether one launch is expected to be faster
@pytest.mark.parametrize("grid, text, one", [
    ((3, 22, 41), 512, True),   # 2706 rows: the text fills the third round
    ((2, 10, 13), 256, False),  # 260 rows
    ((1, 16, 16), 257, True),   # 256 rows: tiles cut along the reduction
    ((3, 20, 20), 512, True),   # 1200 rows
])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("per_token", [False, True])
def test_text_beside_the_self_attention(gpu, monkeypatch, grid, text, one, dtype, per_token):
    from vllm_omni_amd.blocks.wan import WanTransformer3DModel

    rows = grid[0] * grid[1] * grid[2]
    print(f"wan block {dtype} {rows} + {text} rows, per token {per_token}", flush=True)
    assert (_one_launch(rows, text, dtype) == 0) == one
    with torch.inference_mode():
        model = _built(WanTransformer3DModel, dtype, num_layers=1, text_dim=128)
        block = model.blocks[0]
        block.attn2.norm_q.weight.data *= 4  # (a query sees a few text rows instead of the mean of all)
        video = _rand(dtype, 1, 16, grid[0], 2 * grid[1], 2 * grid[2])
        t = torch.full((1, rows) if per_token else (1,), 500.0, device="cuda")
        if per_token:
            t[:, :grid[1] * grid[2]] = 0.0
        x, ctx, temb, mod, rot = model.prepare(video, t, _rand(dtype, 1, text, 128))
        assert x.shape == (1, rows, WIDTH) and ctx.shape == (1, text, WIDTH)
        native = [block(x, ctx, mod, rot).float() for _ in range(2)]
        monkeypatch.setattr(kernels, "NATIVE_BLOCKS", False)
        stepwise = block(x, ctx, mod, rot).float()
    assert torch.equal(native[0], native[1])
    # what the block adds to x. Sums in another order round to a neighbour of the type now and then, at each of a dozen roundings: half a
    # step of the value each, adding up like random ones; a row that is read from a wrong place is off by its whole length
    moved = stepwise - x.float()
    bound = 12 ** 0.5 * (2.0 ** -9 if dtype == torch.bfloat16 else 2.0 ** -12)
    scale = stepwise.norm() / moved.norm()  # (the sum with x is rounded as the whole)
    err = ((native[0] - stepwise).norm() / moved.norm()).item()
    worst = ((native[0] - stepwise).norm(dim=-1) / moved.norm(dim=-1)).max().item()
    print(f"relative difference {err:.2e}, of a row at most {worst:.2e}, bound {bound * max(1.0, scale.item()):.2e}", flush=True)
    assert err <= bound * max(1.0, scale.item()) and worst <= 4 * bound * max(1.0, scale.item())


@pytest.mark.parametrize("rows, text, answer", [
    (2706, 512, 0), (5000, 512, 0),     # the text fills a round that is there anyway
    (8000, 512, -2), (1024, 300, -2),   # two launches are expected to be faster (ODIT_ENOTSUP)
    (2706, 255, -2), (255, 512, -2),    # fewer rows than the tile kernel is chosen for
])
def test_one_launch_where_it_is_expected_to_be_faster(gpu, rows, text, answer):
    assert _one_launch(rows, text, torch.bfloat16) == answer
