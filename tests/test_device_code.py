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
def _assembly(source):
    spec = importlib.util.spec_from_file_location("omni_dit_build_flags", _CSRC / "build.py")
    build = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(build)
    try:
        hipcc = build._hipcc()
    except RuntimeError as e:
        pytest.skip(str(e))
    asm = subprocess.run([hipcc, *build.HIPCC_FLAGS, "--offload-device-only", "-S", str(_CSRC / source), "-o", "-"], capture_output=True,
                         text=True, check=True).stdout
    return [line.split(";")[0].strip() for line in asm.splitlines()]


def _functions(source, labels=False):
    """{kernel: its instructions, one text each, and its labels if asked for} of a translation unit."""
    found, lines = {}, None
    for line in _assembly(source):
        if re.match(r"_Z\w+:$", line):
            lines = found.setdefault(line[:-1], [])
        elif lines is not None and (labels and re.match(r"\.LBB\w+:$", line) or line and not line.startswith(".") and not line.endswith(":")):
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


def _registers(operand):
    m = re.match(r"([sv])(?:\[(\d+):(\d+)\]|(\d+))$", operand)
    if not m:
        return set()
    return {m[1] + str(i) for i in range(int(m[2] or m[4]), int(m[3] or m[4]) + 1)}


def _written_in_front(code, at, scalars, need):
    """The vector instruction, if there is one, that writes one of `scalars` less than `need` wait states in front of `at`, on any way there."""
    while need > 0 and at > 0:
        at -= 1
        text = code[at]
        if text.endswith(":"):
            for i, other in enumerate(code):
                if other.startswith("s_") and "branch" in other and other.split()[1] == text[:-1]:
                    found = _written_in_front(code, i + 1, scalars, need)
                    if found:
                        return found
        elif text.startswith(("s_branch", "s_endpgm")):
            return None
        else:
            if text.startswith("v_") and _registers(text.split()[1].rstrip(",")) & scalars:
                return text
            need -= int(text.split()[1]) + 1 if text.startswith("s_nop") else 1
    return None


@pytest.mark.parametrize("source,states", [("attn_fwd_dma.hip", 0), ("gemm_bf16.hip", 3), ("gemm_bf16_tile.hip", 3), ("gemm_small.hip", 3)])
def test_loads_into_lds_wait_for_their_scalar_registers(source, states):
    """A memory instruction may read a scalar register 5 wait states after a vector instruction has written it and no sooner; for
    the loads in inline assembly the compiler does not see to that. The GEMM kernels' statements wait themselves; attention's
    rest on its descriptors and offsets being formed by scalar instructions."""
    loads = 0
    for name, code in _functions(source, labels=True).items():
        for at, text in enumerate(code):
            if not (text.startswith("buffer_load_dwordx4") and text.endswith("lds")):
                continue
            loads += 1
            scalars = {r for o in re.split(r"[,\s]+", text.replace(", ", " ")) for r in _registers(o) if r[0] == "s"}
            assert len(scalars) >= 4, text
            assert code[at - 2].startswith("s_mov_b32 m0") and code[at - 1] == f"s_nop {states}", (name, code[at - 2:at + 1])
            assert _written_in_front(code, at, scalars, 5) is None, (name, code[at - 8:at + 1])
    assert loads > 50
