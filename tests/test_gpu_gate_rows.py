"""The gate rows of a step in one launch: the bits of the torch expression (one conversion and one product each)."""

import pytest
import torch

from vllm_omni_amd import kernels

pytestmark = pytest.mark.gpu


# 300 projections: more than one launch carries; 97 features and a bias or modulations off 8 bytes: one element a lane
@pytest.mark.parametrize("B,n,C,pad,shift", [(1, 1, 8, 0, 0), (2, 4, 256, 0, 0), (2, 8, 3072, 4, 0), (3, 300, 64, 12, 0), (2, 3, 97, 5, 0),
                                             (1, 5, 1028, 0, 1)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_gate_rows_are_the_bits_of_the_torch_expression(gpu, B, n, C, pad, shift, dtype):
    g = torch.Generator().manual_seed(n)
    mods = torch.randn(B, n * 3 * C + pad, generator=g).to(dtype).cuda()[:, pad:].view(B, n, 3 * C)
    mods[0, 0, 2 * C] = float("inf")
    biases = [torch.randn(C + shift, generator=g).to(dtype).cuda()[shift:] for _ in range(n)]
    with torch.no_grad():
        gates, gated = kernels.gate_rows(mods, biases)
        want = mods[..., 2 * C:].float()
        assert torch.equal(gates, want)
        assert torch.equal(gated, want * torch.stack(biases).float())


def test_what_the_kernel_does_not_take_is_left_to_torch(gpu):
    mods, bias = torch.randn(2, 1, 24, device=gpu).bfloat16(), torch.randn(8, device=gpu).bfloat16()
    with torch.no_grad():
        assert kernels.gate_rows(mods, [bias.float()]) is None          # another type
        assert kernels.gate_rows(mods, [bias[:4]]) is None              # another width
        assert kernels.gate_rows(mods.float(), [bias.float()]) is None
        assert kernels.gate_rows(mods, [bias, bias]) is None            # not 3 C for each
        assert kernels.gate_rows(mods, [None]) is None
        assert kernels.gate_rows(mods.transpose(0, 1), [bias]) is None
    assert kernels.gate_rows(mods, [bias]) is None                      # under autograd
