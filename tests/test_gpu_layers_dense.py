"""One dense tensor through the per-head norm, the rotation or the adaLN alone: the bits that the general kernels give for the same rows with a
stride, for every head size, odd numbers of rows and heads, every type."""

import pytest
import torch

from vllm_omni_amd import kernels
from vllm_omni_amd._lib import ODIT_NORM_HEAD, ODIT_NORM_NONE

pytestmark = pytest.mark.gpu
_TYPES = [torch.bfloat16, torch.float16, torch.float32]


def _strided(x):
    """x [B, S, H, D] as part of wider rows"""
    wide = torch.full((*x.shape[:2], 2 * x.shape[2] * x.shape[3]), float("nan"), dtype=x.dtype, device=x.device)
    view = wide[..., :x.shape[2] * x.shape[3]].unflatten(-1, x.shape[2:])
    view.copy_(x)
    return view


@pytest.mark.parametrize("dtype", _TYPES)
@pytest.mark.parametrize("B,S,H,D", [(1, 77, 24, 128), (2, 33, 5, 64), (1, 1, 1, 8), (3, 7, 2, 256), (1, 513, 1, 32), (2, 16, 3, 16), (1, 5463, 24, 128)])
def test_head_norm(gpu, dtype, B, S, H, D):
    print(f"norm {dtype} {B}x{S}x{H}x{D}", flush=True)
    g = torch.Generator(device=gpu).manual_seed(1)
    x = torch.randn(B, S, H, D, device=gpu, generator=g).to(dtype)
    w = torch.randn(D, device=gpu, generator=g).to(dtype)
    a, b = (torch.full_like(x, float("nan")) for _ in range(2))
    kernels.qknorm_rope(x, None, None, a, None, None, w, None, None, None, eps=1e-6, norm_mode=ODIT_NORM_HEAD)
    kernels.qknorm_rope(_strided(x), None, None, b, None, None, w, None, None, None, eps=1e-6, norm_mode=ODIT_NORM_HEAD)
    assert bool(torch.isfinite(a).all()) and torch.equal(a, b)


@pytest.mark.parametrize("dtype", _TYPES)
@pytest.mark.parametrize("B,S,H,D,rot", [(1, 77, 24, 128, 128), (2, 33, 6, 64, 32), (1, 1, 2, 8, 8), (3, 7, 2, 256, 64), (2, 129, 3, 64, 64), (1, 300, 2, 16, 16)])
def test_rotation(gpu, dtype, B, S, H, D, rot):
    print(f"rotation {dtype} {B}x{S}x{H}x{D} {rot}", flush=True)
    g = torch.Generator(device=gpu).manual_seed(2)
    x = torch.randn(B, S, H, D, device=gpu, generator=g).to(dtype)
    angles = torch.rand(S, rot // 2, device=gpu, generator=g) * 6.28
    a, b = (torch.full_like(x, float("nan")) for _ in range(2))
    for t, out in ((x, a), (_strided(x), b)):
        kernels.qknorm_rope(t, None, None, out, None, None, None, None, angles.cos(), angles.sin(), norm_mode=ODIT_NORM_NONE)
    assert bool(torch.isfinite(a).all()) and torch.equal(a, b)


@pytest.mark.parametrize("dtype", _TYPES)
@pytest.mark.parametrize("B,S,C", [(1, 77, 3072), (3, 5, 256), (2, 1, 512), (2, 9, 1024), (1, 3, 2048), (2, 4, 3080), (1, 5, 4096), (2, 3, 6144), (1, 2, 8192)])
def test_adaln(gpu, dtype, B, S, C):
    if dtype == torch.float32:
        C //= 2
    print(f"adaln {dtype} {B}x{S}x{C}", flush=True)
    g = torch.Generator(device=gpu).manual_seed(3)
    x = torch.randn(B, S, C, device=gpu, generator=g).to(dtype)
    mod = torch.randn(B, 3 * C, device=gpu, generator=g).to(dtype)
    shift, scale, _ = mod.chunk(3, dim=-1)
    wide = torch.full((B, S, 2 * C), float("nan"), dtype=dtype, device=gpu)
    wide[..., :C] = x
    a, b = kernels.adaln_modulate(x, shift, scale, eps=1e-6), kernels.adaln_modulate(wide[..., :C], shift, scale, eps=1e-6)
    assert bool(torch.isfinite(a).all()) and torch.equal(a, b)
