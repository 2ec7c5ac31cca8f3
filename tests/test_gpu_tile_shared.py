"""Tiles that are the sum of two or three sums, parted where the library's kernel that is never run would have parted them."""

import pytest
import torch

from test_gpu_library_kernels import _BOUND, BIAS, FIRST, GATED, GELU, RESIDUAL, _Problem

pytestmark = pytest.mark.gpu


def parted(M, N, K, workers):
    """{(row tile, feature tile): steps at which a sum begins behind its first}, one worker's steps after the other."""
    mt, nt, n = -(-M // 256), -(-N // 256), K // 64
    order = [(r, c) for g in range(0, mt, 16) for c in range(nt) for r in range(g, min(g + 16, mt))]
    if len(order) % workers == 0:
        return {}
    late = order[max(0, len(order) - len(order) % workers - workers):]
    ends, at = set(), 0
    for w in range(workers):
        at += len(late) * n // workers + (w < len(late) * n % workers)
        ends.add(at)
    assert at == len(late) * n
    at = {}
    for e in ends:
        if e % n:
            at.setdefault(late[e // n], set()).add(e % n)
    return at


# (workers: the workspace that the library asks for, in tiles of 256 KB)
@pytest.mark.parametrize("M, N, K, workers, groups", [
    (8192, 9216, 3072, 233, 1),     # workers that are no multiple of 8
    (13202, 5120, 5120, 256, 1),    # a last group of 4 row tiles, 146 rows in the last tile
    (4800, 13824, 5120, 256, 1),    # 4 rounds and two tiles
    (26404, 5120, 5120, 256, 2),    # gates of two groups of rows: each is shared out by itself
    (2400, 5120, 13824, 256, 1),    # fewer tiles than workers: all are parted, some into three
])
def test_where_sums_are_parted(gpu, M, N, K, workers, groups):
    """x = B in step j - 1, 2 in step j and -B behind it, with 2 half a unit of B's last place: 0 in one sum (B + 2 is B), 2 where a sum begins with step j."""
    print(f"parted sums {M}x{N}x{K} groups={groups}", flush=True)
    p = _Problem(gpu, M, N, K, GATED if groups > 1 else BIAS, torch.bfloat16, groups)
    big, n, rows = 2.0 ** 25, K // 64, M // groups
    p.w.fill_(1.0)
    p.gate.fill_(1.0)
    for t in (p.bias, p.gate_bias, p.residual):
        t.zero_()
    found = [{} for _ in range(groups)]
    for j in range(1, n):
        p.x.zero_()
        p.x[:, 64 * (j - 1)] = big
        p.x[:, 64 * j] = 2.0
        p.x[:, 64 * (j + 1) if j + 1 < n else 64 * j + 32] = -big
        out = p.run(FIRST).view(groups, rows, N)
        for g in range(groups):
            corners = out[g, ::256, ::256]
            assert torch.equal(out[g], corners.repeat_interleave(256, 0)[:rows].repeat_interleave(256, 1)[:, :N])
            for r, c in corners.nonzero().tolist():
                assert corners[r, c] == 2.0
                found[g].setdefault((r, c), set()).add(j)
    assert found == [parted(rows, N, K, workers)] * groups


@pytest.mark.parametrize("M, N, K, epilogue, groups", [(4800, 13824, 5120, GELU, 1), (8192, 9216, 3072, RESIDUAL, 1), (13202, 5120, 5120, BIAS, 1), (26404, 5120, 5120, GATED, 2),
                                                      (4800, 5120, 13824, GATED, 2)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_values(gpu, M, N, K, epilogue, groups, dtype):
    p = _Problem(gpu, M, N, K, epilogue, dtype, groups)
    if epilogue == RESIDUAL:
        p.gate.fill_(1.0)  # (it has none)
    out, names = p.names(FIRST)
    assert len(names) == groups and all("gemm_tile_kernel" in n for n in names), names
    y = p.exact()
    assert float((out.double() - y).norm() / y.norm()) < _BOUND[dtype]
    assert torch.equal(out, p.run(FIRST))


def test_order_of_three_sums(gpu):
    """B, 1 and -B in the three sums of a tile, in all orders: 1 where the first two to be added are B and -B (B + 1 is B), which are then the tile's first two."""
    M, N, K, workers = 2400, 5120, 13824, 256
    tiles = {t: sorted(e) for t, e in parted(M, N, K, workers).items() if len(e) == 2}
    assert len(tiles) == 48
    p = _Problem(gpu, M, N, K, BIAS, torch.bfloat16)
    p.bias.zero_()
    for order in ((2.0 ** 25, -(2.0 ** 25), 1.0), (2.0 ** 25, 1.0, -(2.0 ** 25)), (1.0, 2.0 ** 25, -(2.0 ** 25))):
        want, got = torch.full((len(tiles),), 1.0 if order[2] == 1.0 else 0.0), []
        p.x.fill_(1.0)
        # (one reduction element of each sum; a launch for each tile, as those of one column share W)
        for (r, c), (a, b) in tiles.items():
            p.w.zero_()
            for step, v in zip((0, a, b), order):
                p.w[c * 256:c * 256 + 256, 64 * step] = v
            got.append(p.run(FIRST)[r * 256, c * 256].float().cpu())
        assert torch.equal(torch.stack(got), want), (order, got)


def test_a_call_of_two_groups_is_two_calls(gpu):
    p = _Problem(gpu, 26404, 5120, 5120, GATED, torch.bfloat16, 2)
    both = p.run(FIRST).view(2, 13202, 5120)
    for g in range(2):
        one = _Problem(gpu, 13202, 5120, 5120, GATED, torch.bfloat16)
        one.w, one.x, one.residual = p.w, p.x.view(2, 13202, -1)[g], p.residual.view(2, 13202, -1)[g]
        one.gate, one.gate_bias = p.gate[g:g + 1], p.gate_bias[g:g + 1]
        assert torch.equal(one.run(FIRST), both[g])


def test_on_every_replay_of_a_graph(gpu):
    p = _Problem(gpu, 8192, 9216, 3072, BIAS, torch.bfloat16)
    want, side = p.run(FIRST), torch.cuda.Stream()
    torch.cuda.synchronize()
    with torch.cuda.stream(side):
        p.run(FIRST)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=side):
        out = p.run(FIRST)
    for _ in range(3):
        out.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, want) and torch.equal(p.run(FIRST), want)
        torch.cuda.synchronize()
