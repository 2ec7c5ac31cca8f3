"""The waits of test_device_code.py in the tile kernel's forms that round in the library's order. CPU only."""

import re

import pytest

from test_device_code import _functions, _registers, _written_in_front


@pytest.mark.parametrize("unit, forms, sums", [("gemm_tile_apart.hip", 4, 0), ("gemm_tile_shared.hip", 2, 32)])  # (sums: what a lane leaves of a tile)
def test_waits_that_hold_by_statement(unit, forms, sums):
    kernels = _functions(unit, labels=True)
    assert len(kernels) == forms
    for name, code in kernels.items():
        stores = [i for i in code if i.startswith("buffer_store_dwordx4")]
        assert len(stores) >= sums, name
        assert [i for i in stores if not re.search(r"\], 0 offen", i)] == [], name
        loads = [at for at, text in enumerate(code) if text.startswith("buffer_load_dwordx4") and text.endswith("lds")]
        assert loads, name
        for at in loads:
            scalars = {r for o in re.split(r"[,\s]+", code[at]) for r in _registers(o) if r[0] == "s"}
            assert len(scalars) >= 4, code[at]
            assert code[at - 2].startswith("s_mov_b32 m0") and code[at - 1] == "s_nop 3", (name, code[at - 2:at + 1])
            assert _written_in_front(code, at, scalars, 5) is None, (name, code[at - 8:at + 1])
