"""Attention whose running maximum is left behind by one key at a time: a lane holds 4 keys of every 8 for a query, and the maximum over
the lanes of a query is formed only when one of them sees its keys exceed the running one by 2^8. Against a float64 product."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("head_size, keys, queries", [(128, 640, 130), (128, 2112, 33), (64, 640, 130), (64, 193, 1)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_single_keys_take_the_maximum(head_size, keys, queries, dtype):
    from vllm_omni_amd.attention.layer import Attention

    heads, tiles = 8, (keys + 63) // 64
    gen = torch.Generator().manual_seed(head_size + keys)
    q = torch.randn(2, queries, heads, head_size, generator=gen)
    k = torch.randn(2, keys, heads, head_size, generator=gen) * 0.1
    v = torch.randn(2, keys, heads, head_size, generator=gen)
    # in tile j one key, at another place in every tile and head, has a score of about 3 (j + 1) with each query of the positive half space
    unit = torch.ones(head_size) / head_size ** 0.5
    q = q + 4 * unit
    for h in range(heads):
        for j in range(tiles):
            at = min(64 * j + (7 * j + 9 * h) % 64, keys - 1)
            k[:, at, h] = unit * (3.0 * (j + 1)) * head_size ** 0.5 / 4
    q, k, v = (t.to(dtype).cuda() for t in (q, k, v))
    layer = Attention(num_heads=heads, head_size=head_size, causal=False, softmax_scale=head_size ** -0.5, num_kv_heads=heads)
    with torch.inference_mode():
        out = layer(q, k, v, None).double().cpu()
    qd, kd, vd = (t.double().cpu().transpose(1, 2) for t in (q, k, v))
    p = torch.softmax(qd @ kd.transpose(-1, -2) * head_size ** -0.5, dim=-1)
    want = (p @ vd).transpose(1, 2).reshape(out.shape)
    # probabilities and result are each rounded to the type: |error| <= eps (sum p |v| + |result|), and as much again for exp2 and fp32 sums
    eps = torch.finfo(dtype).eps / 2
    bound = 2 * eps * ((p @ vd.abs()).transpose(1, 2).reshape(out.shape) + want.abs()) + 1e-6
    assert bool(((out - want).abs() <= bound).all())


@pytest.mark.parametrize("head_size, keys", [(128, 640), (128, 2112), (64, 193)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_nan_scores_stay_with_their_query(head_size, keys, dtype):
    """A NaN among the queries spoils its own row, one among the keys its head, and one among keys that are excluded nothing."""
    from vllm_omni_amd import kernels

    g = torch.Generator(device="cuda").manual_seed(keys)
    q, k, v = (torch.randn(1, s, 4, head_size, device="cuda", generator=g).to(dtype) for s in (130, keys, keys))
    mask = torch.ones(1, keys, dtype=torch.bool, device="cuda")
    mask[0, 70] = False
    for m in (None, mask):
        clean = kernels.attn_fwd(q, k, v, head_size ** -0.5, key_mask=m)
        spoiled = q.clone()
        spoiled[0, 33, 1, 5] = float("nan")
        out = kernels.attn_fwd(spoiled, k, v, head_size ** -0.5, key_mask=m)
        assert bool(out[0, 33, 1].isnan().all())
        out[0, 33, 1] = clean[0, 33, 1]
        assert torch.equal(out, clean)
        at_key = k.clone()
        at_key[0, 70, 2, 0] = float("nan")
        out = kernels.attn_fwd(q, at_key, v, head_size ** -0.5, key_mask=m)
        if m is None:
            assert bool(out[0, :, 2].isnan().all())
            out[0, :, 2] = clean[0, :, 2]
        assert torch.equal(out, clean)
