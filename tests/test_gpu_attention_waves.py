"""Head size 128 with 4 wavefronts or 8 to a workgroup (csrc/attn_fwd_dma.hip, dma_waves): the form that a launch has, the bits of
the same heads in launches of the other one, and the result in 64 bits."""

import pytest
import torch

from vllm_omni_amd import kernels

# (queries, keys, heads of one batch row) on 256 compute units, units being of 128 queries
CASES = [
    (300, 1984, 2, 4),     # 31 key tiles
    (130, 1985, 3, 4),     # 32: few units, cut by keys
    (256, 2100, 33, 8),    # 66 units, whole pairs
    (256, 2100, 32, 4),    # 64: one on every fourth compute unit
    (384, 2100, 32, 4),    # 96, no pairs
    (256, 2050, 65, 4),    # 130: too many to be cut
    (512, 2050, 65, 8),    # 260: two units on some compute units
    (513, 2050, 65, 4),    # 325, no pairs
    (512, 2050, 97, 4),    # 388: more than one and a half for each
    (257, 4033, 8, 4),     # 64 key tiles
    (1024, 4033, 129, 8),  # and more than two rounds
    (1024, 4033, 128, 4),  # two
    (200, 8128, 2, 4),     # 127 key tiles
    (200, 8129, 2, 8),     # 128
]


@pytest.mark.parametrize("Sq,Sk,H,waves", CASES)
def test_form(Sq, Sk, H, waves):
    if torch.cuda.is_available() and torch.cuda.get_device_properties(0).multi_processor_count != 256:
        pytest.skip("the sizes are for 256 compute units")
    assert f"attn_fwd_dma_kernel<T, 128, {waves}, 0>" in kernels.attn_plan(1, Sq, Sk, H, 128)


@pytest.mark.gpu
@pytest.mark.parametrize("Sq,Sk,H,waves", CASES)
@pytest.mark.parametrize("dtype,masked", [(torch.bfloat16, False), (torch.float16, True)])
def test_bits_and_result(gpu, Sq, Sk, H, waves, dtype, masked):
    print(f"attention {dtype} Sq={Sq} Sk={Sk} H={H} masked={masked}", flush=True)
    g = torch.Generator(device=gpu).manual_seed(Sq + Sk)
    q, k, v = (torch.randn(1, s, H, 128, generator=g, device=gpu).to(dtype) for s in (Sq, Sk, Sk))
    scale = 128 ** -0.5
    mask = (torch.rand(1, Sk, generator=g, device=gpu) < 0.7) if masked else None
    whole = kernels.attn_fwd(q, k, v, scale, key_mask=mask, use_workspace=False)
    for h in range(0, H, max(1, H // 5)):
        one = [t[:, :, h:h + 1] for t in (q, k, v)]
        assert torch.equal(whole[:, :, h:h + 1], kernels.attn_fwd(*one, scale, key_mask=mask, use_workspace=False))
    cut = kernels.attn_fwd(q, k, v, scale, key_mask=mask)
    heads, rows = sorted({0, H // 2, H - 1}), sorted({0, Sq // 2, Sq - 1})
    qd, kd, vd = (t.double().cpu().transpose(1, 2) for t in (q[:, rows][:, :, heads], k[:, :, heads], v[:, :, heads]))
    s = (qd @ kd.transpose(-1, -2).contiguous()) * scale
    if masked:
        s = s.masked_fill(~mask.cpu()[:, None, None, :], float("-inf"))
    want = (torch.softmax(s, dim=-1) @ vd).transpose(1, 2)
    # probabilities (which sum to one) and the result are rounded to the type once each: half a step of |v| each, and 1e-3 for the
    # float32 scores
    tol = (2 * 0.5 * (2.0 ** -7 if dtype == torch.bfloat16 else 2.0 ** -10) + 1e-3) * v.abs().max().item()
    for o in (whole, cut):
        assert (o[:, rows][:, :, heads].double().cpu() - want).abs().max().item() < tol
