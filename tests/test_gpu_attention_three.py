"""Head size 64 with three workgroups per compute unit and, where those need as many rounds, with two (csrc/attn_fwd_dma.hip,
fills_two): the bits of the same attention in launches of fewer units, and the result in 64 bits."""

import pytest
import torch

from vllm_omni_amd import kernels

pytestmark = pytest.mark.gpu


# units of 128 query rows: from 769 to 1024 a launch runs two workgroups per compute unit
@pytest.mark.parametrize("B,Sq,Sk,H,Hkv,masked", [
    (1, 5500, 1, 16, 16, False),    # one key
    (1, 5500, 65, 16, 4, False),    # 688 units, a tile and one key
    (1, 2049, 300, 31, 31, False),  # 527 units, one row in the last block, keys too few to be split
    (1, 1300, 64, 48, 48, False),   # 528 units, one tile
    (2, 1536, 130, 32, 32, False),  # 768 units: all there is room for
    (1, 6145, 1100, 16, 16, False), # 784 units: two workgroups per compute unit
    (1, 8192, 64, 16, 4, False),    # 1024 units: the last launch of two
    (3, 700, 700, 40, 8, True),     # batch rows spread over the XCDs
    (2, 1357, 129, 31, 31, True),   # heads that do not divide over them
    (2, 2049, 300, 24, 24, True),   # 816 units: two with mask words, batch rows spread over the XCDs
    (2, 2049, 65, 25, 25, True),    # 850 units, heads that do not divide over them
    (3, 1200, 193, 40, 8, True),    # 1200 units: three again
])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_three_workgroups_per_compute_unit(gpu, B, Sq, Sk, H, Hkv, masked, dtype):
    print(f"attention {dtype} B={B} Sq={Sq} Sk={Sk} H={H}/{Hkv} masked={masked}", flush=True)
    g = torch.Generator().manual_seed(Sq + Sk)
    q, k, v = (torch.randn(B, s, h, 64, generator=g).to(dtype).cuda() for s, h in ((Sq, H), (Sk, Hkv), (Sk, Hkv)))
    mask = None
    if masked:
        mask = torch.arange(Sk, device=gpu)[None, :] < torch.tensor([Sk, max(1, Sk // 3), Sk - 1][:B], device=gpu)[:, None]
    for ws in (True, False):
        o, lse = kernels.attn_fwd(q, k, v, 0.125, key_mask=mask, return_lse=True, use_workspace=ws)
        per = H // Hkv
        for h0 in range(0, Hkv, max(1, Hkv // 4)):  # a quarter of the heads, one batch row at a time: well below 513 units
            hk = slice(h0, min(h0 + max(1, Hkv // 4), Hkv))
            hq = slice(hk.start * per, hk.stop * per)
            for b in range(B):
                ob, lb = kernels.attn_fwd(q[b:b + 1, :, hq], k[b:b + 1, :, hk], v[b:b + 1, :, hk], 0.125,
                                          key_mask=None if mask is None else mask[b:b + 1], return_lse=True, use_workspace=False)
                assert torch.equal(o[b:b + 1, :, hq], ob) and torch.equal(lse[b:b + 1, hq], lb)
    rows = torch.tensor([0, Sq // 2, Sq - 1])
    qd, kd, vd = (t.double().cpu().transpose(1, 2) for t in (q[:, rows.to(gpu)], k.repeat_interleave(H // Hkv, 2), v.repeat_interleave(H // Hkv, 2)))
    s = (qd @ kd.transpose(-1, -2).contiguous()) * 0.125
    if masked:
        s = s.masked_fill(~mask.cpu()[:, None, None, :], float("-inf"))
    want = (torch.softmax(s, dim=-1) @ vd).transpose(1, 2)
    # probabilities (which sum to one) and the result are rounded to the type once each: half a step of |v| each, and 1e-3 for the
    # float32 scores
    tol = (2 * 0.5 * (2.0 ** -7 if dtype == torch.bfloat16 else 2.0 ** -10) + 1e-3) * v.abs().max().item()
    assert (o[:, rows.to(gpu)].double().cpu() - want).abs().max().item() < tol
