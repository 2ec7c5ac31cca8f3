"""Waits that hold by statement: the assembly of the kernels that move data with inline assembly or raw buffer instructions, as the
compiler makes it here from their sources, looked through for what the hardware leaves to the program. CPU only."""

import functools
import importlib.util
import re
import subprocess
from pathlib import Path

import pytest

_CSRC = Path(__file__).resolve().parents[1] / "vllm-omni_amd" / "csrc"


@functools.lru_cache(maxsize=None)
def _functions(source):
    """{kernel: its instructions, one text each} of a translation unit; labels and directives are left out."""
    spec = importlib.util.spec_from_file_location("omni_dit_build_flags", _CSRC / "build.py")
    build = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(build)
    try:
        hipcc = build._hipcc()
    except RuntimeError as e:
        pytest.skip(str(e))
    asm = subprocess.run([hipcc, *build.HIPCC_FLAGS, "--offload-device-only", "-S", str(_CSRC / source), "-o", "-"], capture_output=True,
                         text=True, check=True).stdout
    found, lines = {}, None
    for line in asm.splitlines():
        line = line.split(";")[0].strip()
        if re.match(r"_Z\w+:$", line):
            lines = found.setdefault(line[:-1], [])
        elif line and lines is not None and not line.startswith(".") and not line.endswith(":"):
            lines.append(line)
    return {k: v for k, v in found.items() if any(i.startswith("s_endpgm") for i in v)}


def test_partial_tiles_are_stored_without_a_scalar_offset():
    """A vector instruction may write a 16-byte store's data registers 2 wait states behind it and no sooner. The compiler sees to
    that unless the store has its offset in a scalar register."""
    kernels = _functions("gemm_bf16_tile.hip")
    assert len(kernels) == 4
    for name, code in kernels.items():
        stores = [i for i in code if i.startswith("buffer_store_dwordx4")]
        assert len(stores) >= 16, name  # 4 quadrants of 4 or 8, and those of a part that gives up
        assert [i for i in stores if not re.search(r"\], 0 offen", i)] == [], name


def test_small_kernel_waits_for_its_reads_at_every_barrier():
    """Behind a step's barrier the stage that was read in the step before is refilled: the wait in front of the barrier names the
    reads too, wherever the matrix instructions that use them end up."""
    kernels = _functions("gemm_small.hip")
    assert len(kernels) == 8
    for name, code in kernels.items():
        barriers = [i for i, text in enumerate(code) if text.startswith("s_barrier")]
        assert barriers, name
        for at in barriers:
            wait = next(text for text in reversed(code[:at]) if text.startswith("s_waitcnt"))
            assert "lgkmcnt(0)" in wait and "vmcnt" in wait, (name, code[at - 6:at + 1])
