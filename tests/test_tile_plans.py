"""Plans of the tile kernel, by the library's own function: how its GPU tests' problems are cut, and where rows of padding are fetched from. CPU only."""

import subprocess
from pathlib import Path

import pytest

from test_gpu_gemm_tile_parts import HEADS, PARTS
from test_gpu_tile_shared import parted

_ROOT = Path(__file__).resolve().parents[1]


@pytest.fixture(scope="module")
def ask(tmp_path_factory):
    pkg, exe = _ROOT / "vllm-omni_amd", tmp_path_factory.mktemp("plan") / "plan_host"
    if not (pkg / "libomni_dit_hip.so").exists():
        pytest.skip("the library is not built")
    subprocess.run(["hipcc", "-x", "hip", "--offload-host-only", "-O1", "-std=c++17", f"-I{pkg / 'csrc'}", str(_ROOT / "tests" / "native" / "plan_host.cpp"), "-o", str(exe),
                    f"-L{pkg}", "-l:libomni_dit_hip.so", f"-Wl,-rpath,{pkg}"], check=True, capture_output=True)

    def ask(*lines):
        out = subprocess.run([str(exe)], input="\n".join(" ".join(map(str, line)) for line in lines) + "\n", text=True, check=True, capture_output=True).stdout
        return [tuple(map(int, line.split())) for line in out.splitlines()]

    return ask


def test_problems_of_the_parts_tests(ask):
    """128 rows to a tile, none of them whole, in as many parts as the tests say."""
    assert ask(*((M, N, K) for M, N, K, _ in PARTS)) == [(128, parts, 0) for *_, parts in PARTS]
    assert ask(*((S0, S1, 3 * 128 * H, K) for S0, S1, H, K, _ in HEADS)) == [(128, parts, 0) for *_, parts in HEADS]


def test_more_than_four_parts_only_of_low_tiles_without_whole_ones(ask):
    plans = ask(*((M, N, K) for M in range(100, 3000, 37) for N in (8, 512, 3072, 9216) for K in (64, 704, 3072, 12288)))
    assert {p for _, p, _ in plans} == {1, 2, 3, 4, 5, 6, 7, 8}
    assert all(parts <= 4 or (bm == 128 and whole == 0) for bm, parts, whole in plans)


# up to 2^32 bytes, to the last row of the tile and the last element of the reduction: their own place; from there on the operand's last row
@pytest.mark.parametrize("rows, tile, K", [(1025, 256, 64), (1024, 256, 64), (130, 128, 3072)])
def test_where_rows_of_padding_are_fetched_from(ask, rows, tile, K):
    end = -(-rows // tile) * tile
    fits = (2**31 - K - 1) // end  # the longest row
    assert ask(("pad", rows, tile, K, K), ("pad", rows, tile, fits, K), ("pad", rows, tile, fits + 1, K), ("pad", rows, tile, 2**40, K)) == [(end,), (end,), (rows - 1,), (rows - 1,)]


def test_shares_of_tiles(ask):
    """Where the shares of TileShares part a tile is where workers that take one step after the other do."""
    problems = [(M, N, K, w) for M in (8192, 8193, 13202, 20011) for N in (3072, 5120, 9216) for K in (64, 448, 5120) for w in (1, 7, 233, 256)] + [(2400, 5120, 13824, 256), (1500, 5120, 13824, 206)]
    answers = ask(*(("shares", *p) for p in problems))
    for (M, N, K, w), (known, tiles, first, share, more) in zip(problems, answers):
        mt, nt, n = -(-M // 256), -(-N // 256), K // 64
        order = [(r, c) for g in range(0, mt, 16) for c in range(nt) for r in range(g, min(g + 16, mt))]
        assert known == 1 and tiles == len(order)
        ends = [i * share + min(i, more) for i in range(1, w + 1)] if share else []
        assert {(order[first + e // n], e % n) for e in ends if e % n} == {(t, e) for t, es in parted(M, N, K, w).items() for e in es}
        assert not share or (ends[-1] == (tiles - first) * n and first % w == 0 and (tiles < w or n <= share))
    assert [a[0] for a in ask(("shares", 256, 2560, 64, 11), ("shares", 256, 2560, 64, 0))] == [0, 0]  # (a worker without a step, no workers)
