"""The waits of test_device_code.py in the forms of the GEMM kernels that end in query, key and value heads. CPU only."""

import re

import pytest

from test_device_code import _functions, _written_in_front, _registers


def test_partial_tiles_are_stored_without_a_scalar_offset():
    kernels = _functions("gemm_tile_heads.hip")
    assert len(kernels) == 4
    for name, code in kernels.items():
        stores = [i for i in code if i.startswith("buffer_store_dwordx4")]
        assert len(stores) >= 16, name
        assert [i for i in stores if not re.search(r"\], 0 offen", i)] == [], name


def test_small_kernel_waits_for_its_reads_at_every_barrier():
    kernels = _functions("gemm_small_heads.hip")
    assert len(kernels) == 8
    for name, code in kernels.items():
        barriers = [i for i, text in enumerate(code) if text.startswith("s_barrier")]
        assert len(barriers) >= 2, name  # a step's, and the one behind the squares
        for at in barriers:
            wait = next(text for text in reversed(code[:at]) if text.startswith("s_waitcnt"))
            assert "lgkmcnt(0)" in wait and "vmcnt" in wait, (name, code[at - 6:at + 1])


@pytest.mark.parametrize("source", ["gemm_tile_heads.hip", "gemm_small_heads.hip"])
def test_loads_into_lds_wait_for_their_scalar_registers(source):
    loads = 0
    for name, code in _functions(source, labels=True).items():
        for at, text in enumerate(code):
            if text.startswith("buffer_load_dwordx4") and text.endswith("lds"):
                loads += 1
                scalars = {r for o in re.split(r"[,\s]+", text) for r in _registers(o) if r[0] == "s"}
                assert len(scalars) >= 4, text
                assert code[at - 2].startswith("s_mov_b32 m0") and code[at - 1] == "s_nop 3", (name, code[at - 2:at + 1])
                assert _written_in_front(code, at, scalars, 5) is None, (name, code[at - 8:at + 1])
    assert loads > 16
