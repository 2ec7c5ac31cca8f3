"""GELU(tanh) in the hand-written GEMMs' epilogue over every finite value of the type, against float64: an identity weight
hands each value to the epilogue exactly."""

import pytest
import torch

from vllm_omni_amd import kernels

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype,repeat", [(torch.float16, 1), (torch.bfloat16, 1), (torch.bfloat16, 5)])  # (5: the kernel for many rows)
def test_gelu_epilogue_rounds_like_float64(gpu, dtype, repeat):
    bits = torch.arange(-32768, 32768, dtype=torch.int32).to(torch.int16)
    x = bits.view(dtype)
    # (values whose square overflows float32 make the exponent infinite, which is part of the range)
    x = torch.where(x.isfinite(), x, torch.zeros_like(x)).view(256, 256).repeat(repeat, 1)
    out = kernels.linear(x.to(gpu), torch.eye(256).to(dtype).to(gpu), None, activation="gelu_tanh", engine="handwritten").cpu()
    d = x.double()
    want64 = d / (1 + torch.exp(-2 * 0.7978845608028654 * (d + 0.044715 * d ** 3)))
    want = want64.to(dtype)
    assert torch.equal(out.isfinite(), want.isfinite())
    # float32's relative error (1e-5 where the result is tiny, 2e-6 elsewhere) can only move a result that lies that close to
    # the middle between two neighbours: one step of the type, and rarely
    step = (out.view(torch.int16).int() - want.view(torch.int16).int()).abs()
    same = (step == 0) | ((out == 0) & (want == 0))
    # below 2^-122 the sigmoid's reciprocal is no normal float32 (x down to -10, sigmoid below 2^-126): flushed to zero or not
    tiny = (want64.abs() < 2.0 ** -122) & (out.double().abs() < 2.0 ** -122)
    assert (same | tiny | (step == 1)).all()
    share = (~(same | tiny)).float().mean().item()
    print(f"{dtype} x{repeat}: {share:.2e} of the values one step off", flush=True)
    assert share <= 2e-3
    zero = x == 0
    assert (out[zero] == 0).all()
