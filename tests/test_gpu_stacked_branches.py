"""The two branches of classifier-free guidance stacked, padded and masked in one launch, against torch's concatenations."""

import pytest
import torch

from vllm_omni_amd import _lib, denoise, kernels
from vllm_omni_amd.blocks.qwen_image import joint_key_mask

pytestmark = pytest.mark.gpu


# (rows of 1, 2, 4, 8 and 16 byte granules; one workgroup's 1024 granules, one more, one less)
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("shapes", [((1,), (1,)), ((5,), (5,)), ((1, 171, 3584), (1, 23, 3584)), ((1, 23, 64), (1, 171, 64)), ((2, 7, 3), (2, 9, 3)), ((3, 1, 4), (3, 6, 4)),
                                    ((1, 1024, 8), (1, 1023, 8)), ((2, 1025, 1), (2, 1, 1)), ((2, 5), (2, 5)), ((1, 2, 3, 5), (1, 4, 3, 5))])
def test_stacked(gpu, dtype, shapes):
    torch.manual_seed(1)
    p, n = (torch.randn(s, device=gpu).to(dtype) for s in shapes)
    pm, nm = (torch.rand(s[:2], device=gpu) < 0.5 for s in shapes)
    pairs = [(p, n)] + ([(p, n, None, None), (p, n, pm, None), (p, n, None, nm), (p, n, pm, nm)] if p.dim() > 1 else [])
    with torch.inference_mode():
        got = kernels.stack_pairs(pairs)
        want = [denoise._stacked(pair) for pair in pairs]
    assert all(torch.equal(a, b) and a.dtype == b.dtype for a, b in zip(got, want, strict=True))


def test_not_stacked(gpu):
    x, other = torch.randn(2, 4, 8, device=gpu), torch.randn(2, 4, 6, device=gpu)
    with torch.inference_mode():
        assert kernels.stack_pairs([(x, x)]) is not None
        for pair in ((x, other), (x, x.half()), (x, x.cpu()), (x, x.transpose(1, 2)), (x, None), (x, x[:1]), (x[:, :0], x), (x, x, None, torch.ones(2, 4, device=gpu)),
                     (x, x, torch.ones(2, 3, device=gpu, dtype=torch.bool), None), (x.long(), x.long())):
            assert kernels.stack_pairs([(x, x), pair]) is None
        assert kernels.stack_pairs([(x, x)] * 9) is None
    assert kernels.stack_pairs([(x, x)]) is None  # with gradients: torch's concatenation has a backward
    piece = (_lib.PadPiece * 2)()
    lib = _lib.load()
    assert lib.odit_pad_rows(piece, 17, None) == -1 and lib.odit_pad_rows(piece, 2, None) == -1 and lib.odit_pad_rows(None, 0, None) == 0


@pytest.mark.parametrize("B,S,more", [(1, 171, 1024), (2, 1, 1), (3, 64, 4096), (2, 77, 0), (2, 500, 3000)])
def test_joint_mask(gpu, B, S, more):
    mask = torch.rand(B, S, device=gpu) < 0.5
    want = torch.cat([mask, torch.ones(B, more, device=gpu, dtype=torch.bool)], dim=1)
    with torch.inference_mode():
        assert torch.equal(kernels.extend_mask(mask, more), want)
        for m in (mask, mask.long(), mask[:1].expand(B, S), torch.cat([mask, mask], 1)[:, :S]):
            assert torch.equal(joint_key_mask(m, None, B, S, more, mask.device), torch.cat([m.bool(), want[:, S:]], dim=1))
