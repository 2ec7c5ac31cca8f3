"""A model of a few hundred channels: gates and biases as they are give the bits of gate and gate * bias rows, and whether a block's products are
the small kernel's is answered as the launches are made."""

import pytest
import torch

from vllm_omni_amd import _lib, kernels
from vllm_omni_amd.blocks.qwen_image import QwenImageTransformer2DModel

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("heads,head_dim,axes,B,grid,txt", [(4, 64, (8, 28, 28), 1, (16, 16), 64), (4, 64, (8, 28, 28), 2, (5, 7), 9),
                                                            (3, 128, (16, 56, 56), 2, (12, 9), 33), (6, 64, (8, 28, 28), 1, (40, 40), 20)])
def test_without_gate_rows(gpu, monkeypatch, dtype, heads, head_dim, axes, B, grid, txt):
    print(f"small model {dtype} {heads}x{head_dim} B={B} {grid} + {txt}", flush=True)
    g = torch.Generator(device=gpu).manual_seed(5)
    model = QwenImageTransformer2DModel(num_layers=2, attention_head_dim=head_dim, num_attention_heads=heads, joint_attention_dim=256,
                                        axes_dims_rope=axes).to(device=gpu, dtype=dtype)
    with torch.no_grad():
        for p in model.parameters():
            p.normal_(0.0, 0.05, generator=g)
    model.fuse_modulation()
    args = dict(hidden_states=torch.randn(B, grid[0] * grid[1], 64, device=gpu, generator=g).to(dtype),
                encoder_hidden_states=torch.randn(B, txt, 256, device=gpu, generator=g).to(dtype),
                timestep=torch.full((B,), 0.7, device=gpu, dtype=dtype), img_shapes=[[(1, *grid)]] * B, txt_seq_lens=[txt] * B, return_dict=False)
    made = []
    rows = kernels.gate_rows
    monkeypatch.setattr(kernels, "gate_rows", lambda *a: made.append(1) or rows(*a))
    with torch.inference_mode():
        got = model(**args)[0]
        left_out = not made
        assert left_out == kernels.small_pairs((B * grid[0] * grid[1], B * txt), (heads * head_dim,) * 2, (heads * head_dim, 4 * heads * head_dim))
        monkeypatch.setattr(kernels, "small_pairs", lambda *a: False)
        want = model(**args)[0]
    assert made and bool(torch.isfinite(want).all()) and torch.equal(got, want)


@pytest.mark.parametrize("M0,M1,N,K", [(256, 64, 256, 1024), (256, 64, 256, 256), (1024, 128, 256, 1024), (64, 64, 2048, 2048), (64, 64, 4096, 2048),
                                       (8, 1, 128, 128), (8, 8, 64, 128), (128, 128, 256, 2112), (128, 20, 520, 192), (8192, 512, 256, 256)])
def test_the_answer_is_the_launch(gpu, M0, M1, N, K):
    """A launch of the kernel for small products needs no workspace: with none, a pair is launched exactly where it is that kernel's."""
    C, dtype = _lib.C, torch.bfloat16
    x, w = [torch.randn(m, K, device=gpu, dtype=dtype) for m in (M0, M1)], torch.randn(N, K, device=gpu, dtype=dtype)
    out = [torch.zeros(m, N, device=gpu, dtype=dtype) for m in (M0, M1)]
    q = (_lib.LinearProblem * 2)()
    for p, a, o in zip(q, x, out):
        p.x, p.w, p.out, p.M, p.ldx, p.ldw, p.ldo = a.data_ptr(), w.data_ptr(), o.data_ptr(), a.shape[0], K, K, N
    lib = _lib.load()
    with torch.profiler.profile(activities=[torch.profiler.ProfilerActivity.CUDA]) as prof:
        rc = lib.odit_linear_pair(C.addressof(q), N, K, _lib.ODIT_EPI_NONE, 0, 0, 0, None, 0, torch.cuda.current_stream().cuda_stream)
        torch.cuda.synchronize()
    small = rc == 0 and any("gemm_small_kernel" in e.key for e in prof.key_averages())
    assert bool(lib.odit_linear_pair_is_small(M0, M1, N, K)) == small
