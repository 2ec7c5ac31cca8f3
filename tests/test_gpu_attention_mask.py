"""Key masks of the attention kernel: a mask with no excluded key gives the bits of no mask, any other one the attention over
the keys it leaves, whichever way the kernel holds the mask (words per key tile, or bytes past 65536 keys)."""

import pytest
import torch

from vllm_omni_amd import kernels

pytestmark = pytest.mark.gpu


def _qkv(B, Sq, Sk, H, D, dtype, seed=0):
    g = torch.Generator().manual_seed(seed)
    return tuple(torch.randn(B, s, H, D, generator=g).to(dtype).cuda() for s in (Sq, Sk, Sk))


# 16640 queries x 4 heads: 520 units of 128 rows, eight more than run at once, whose keys are split in two ranges
@pytest.mark.parametrize("B,Sq,Sk,H,D", [(2, 70, 1, 2, 64), (2, 70, 63, 2, 128), (1, 33, 64, 1, 64), (2, 200, 1000, 3, 128),
                                         (1, 300, 2112, 2, 128), (1, 16640, 1100, 4, 64), (1, 33, 65536, 1, 64), (1, 33, 65669, 1, 128)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_all_true_mask_gives_the_bits_of_no_mask(gpu, B, Sq, Sk, H, D, dtype):
    q, k, v = _qkv(B, Sq, Sk, H, D, dtype)
    mask = torch.ones(B, Sk, dtype=torch.bool, device=gpu)
    for ws in (True, False):
        o, lse = kernels.attn_fwd(q, k, v, D ** -0.5, return_lse=True, use_workspace=ws)
        om, lm = kernels.attn_fwd(q, k, v, D ** -0.5, key_mask=mask, return_lse=True, use_workspace=ws)
        assert torch.equal(o, om) and torch.equal(lse, lm)


def _masks(Sk, n_rows):
    """Padding at the edges of 64-key tiles, tiles that are excluded as a whole, single keys, and a row without any key."""
    rows = [torch.arange(Sk) < n for n in (1, 63, 64, 65, 127, 128, 129, Sk - 1, Sk) if 0 < n <= Sk]
    a = torch.arange(Sk)
    rows += [a >= min(64, Sk - 1), (a < 64) | (a >= 128), a % 2 == 0, a == Sk - 1, (a // 64) % 2 == 1, a < 0,
             torch.rand(Sk, generator=torch.Generator().manual_seed(1)) < 0.5]
    return torch.stack(rows)


def _reference(q, k, v, mask, scale):
    """float64 on the CPU, row by row of the batch."""
    q, k, v = (t.double().cpu().transpose(1, 2) for t in (q, k, v))
    s = (q @ k.transpose(-1, -2).contiguous()) * scale
    s = s.masked_fill(~mask.cpu()[:, None, None, :], float("-inf"))
    lse = torch.logsumexp(s, dim=-1)
    p = torch.exp(s - torch.where(lse.isinf(), torch.zeros_like(lse), lse)[..., None])
    return (p @ v).transpose(1, 2), lse


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("Sk", [64, 130, 449])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_masked_attention_against_float64(gpu, Sk, D, dtype):
    mask = _masks(Sk, None)
    B = mask.shape[0]
    q, k, v = _qkv(B, 37, Sk, 2, D, dtype)
    want, want_lse = _reference(q, k, v, mask, D ** -0.5)
    o, lse = kernels.attn_fwd(q, k, v, D ** -0.5, key_mask=mask.to(gpu), return_lse=True)
    # probabilities (which sum to one) and the result are rounded to the type once each: half a step of |v| each, and 1e-3
    # for the float32 scores
    tol = (2 * 0.5 * (2.0 ** -7 if dtype == torch.bfloat16 else 2.0 ** -10) + 1e-3) * v.abs().max().item()
    assert (o.double().cpu() - want).abs().max().item() <= tol
    dead = ~mask.any(dim=1)
    assert dead.any() and (o[dead.to(gpu)] == 0).all() and (lse[dead.to(gpu)] == float("-inf")).all()
    assert (lse.double().cpu() - want_lse)[~dead].abs().max().item() <= 1e-3


@pytest.mark.parametrize("Sk", [65536, 65669])
def test_padding_equals_shorter_keys_at_the_longest_word_table_and_past_it(gpu, Sk):
    q, k, v = _qkv(1, 33, Sk, 1, 64, torch.bfloat16)
    live = 64 * 20 + 17
    mask = (torch.arange(Sk, device=gpu) < live)[None]
    o = kernels.attn_fwd(q, k, v, 0.125, key_mask=mask)
    want = kernels.attn_fwd(q, k[:, :live].contiguous(), v[:, :live].contiguous(), 0.125)
    # the tiles behind the last key add exact zeros; the key-split of the launch may differ: one step of the type
    torch.testing.assert_close(o.float(), want.float(), rtol=2.0 ** -7, atol=2.0 ** -9)


# A unit ends with its last tile that has a live key. 130 and 71 key tiles: the search for it goes over several windows of 64
# tiles, empty ones among them; 8 heads x 700 queries: batch rows shared out over the XCDs; 16640 queries: a last round cut along the keys, whose
# ranges may hold no live key; heads of 128 over 2048 keys and more: workgroups of eight wavefronts.
@pytest.mark.parametrize("B,Sq,Sk,H,Hkv,D", [(6, 40, 8257, 2, 1, 64), (6, 300, 4500, 1, 1, 128), (6, 700, 1024, 8, 2, 64),
                                             (1, 16640, 1100, 4, 4, 64), (6, 700, 2049, 8, 8, 128)])
def test_units_end_with_their_last_live_tile(gpu, B, Sq, Sk, H, Hkv, D):
    g = torch.Generator().manual_seed(Sk)
    q = torch.randn(B, Sq, H, D, generator=g).bfloat16().cuda()
    k, v = (torch.randn(B, Sk, Hkv, D, generator=g).bfloat16().cuda() for _ in range(2))
    a = torch.arange(Sk)
    n = (Sk + 63) // 64
    some = torch.rand(n, generator=g) < 0.1
    some[n // 2] = True
    rows = [a >= Sk - 70, (a >= 64) & (a < 128 + 5), some[a // 64] & (a % 3 == 0), a == Sk // 2, a < 0, a // 64 != 1]
    mask = torch.stack([rows[(Sk + i) % 6] for i in range(B)])
    rep = H // Hkv
    want, want_lse = _reference(q, k.repeat_interleave(rep, 2), v.repeat_interleave(rep, 2), mask, D ** -0.5)
    tol = (2 * 0.5 * 2.0 ** -7 + 1e-3) * v.abs().max().item()  # as above
    for ws in (True, False):
        o, lse = kernels.attn_fwd(q, k, v, D ** -0.5, key_mask=mask.cuda(), return_lse=True, use_workspace=ws)
        assert (o.double().cpu() - want).abs().max().item() <= tol
        dead = ~mask.any(dim=1)
        assert (o[dead.cuda()] == 0).all() and (lse[dead.cuda()] == float("-inf")).all()
        if not dead.all():
            assert (lse.double().cpu() - want_lse)[~dead].abs().max().item() <= 1e-3
