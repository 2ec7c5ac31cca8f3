"""One tensor through the norm and rotary kernel: with an even number of heads a lane takes the same vector of both halves of a
row, with an odd number one vector. Heads do not depend on each other, so one launch over H heads gives the bits of H launches
over one head each."""

import pytest
import torch

from vllm_omni_amd import kernels
from vllm_omni_amd._lib import ODIT_NORM_HEAD, ODIT_NORM_NONE

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B,S,H,D,rot", [(1, 1, 2, 64, 64), (2, 77, 6, 64, 32), (2, 33, 3, 128, 128), (1, 129, 24, 128, 128), (3, 5, 40, 32, 16)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("norm_mode", [ODIT_NORM_NONE, ODIT_NORM_HEAD])
@pytest.mark.parametrize("neox,ref_rounding", [(False, False), (True, False), (False, True), (True, True)])
def test_all_heads_of_one_tensor_give_the_bits_of_single_heads(gpu, B, S, H, D, rot, dtype, norm_mode, neox, ref_rounding):
    g = torch.Generator().manual_seed(S)
    x = torch.randn(B, S, H, D, generator=g).to(dtype).cuda()
    w = torch.randn(D, generator=g).to(dtype).cuda() if norm_mode == ODIT_NORM_HEAD else None
    a = torch.rand(S, rot // 2, generator=g).cuda() * 6.28
    kw = dict(norm_mode=norm_mode, neox=neox, ref_rounding=ref_rounding)
    out = torch.full((B, S + 3, H, D), 7.0, dtype=dtype, device=gpu)
    kernels.qknorm_rope(x, None, None, out, None, None, w, None, a.cos(), a.sin(), out_seq_offset=2, **kw)
    assert (out[:, :2] == 7).all() and (out[:, S + 2:] == 7).all()
    for h in range(H):
        one = torch.empty(B, S, 1, D, dtype=dtype, device=gpu)
        kernels.qknorm_rope(x[:, :, h:h + 1].contiguous(), None, None, one, None, None, w, None, a.cos(), a.sin(), **kw)
        assert torch.equal(out[:, 2:S + 2, h:h + 1], one)
    inplace = x.clone()
    kernels.qknorm_rope(inplace, None, None, inplace, None, None, w, None, a.cos(), a.sin(), **kw)
    assert torch.equal(inplace, out[:, 2:S + 2])
