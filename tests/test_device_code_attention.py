"""What the attention kernel's launch rules and inline assembly rest on, read from the assembly that the compiler makes here of
attn_fwd_dma.hip. CPU only."""

import re

import pytest

from test_device_code import _CSRC, _assembly


def _kernels():
    """{(element type, D, wavefronts, form): its kernel descriptor} of every instantiation."""
    found, at = {}, None
    for line in _assembly("attn_fwd_dma.hip"):
        m = re.match(r"\.amdhsa_kernel \w*attn_fwd_dma_kernelINS_\d(b?f16)_tELi(\d+)ELi(\d)ELi(\d)E", line)
        if m:
            at = found.setdefault((m[1], int(m[2]), int(m[3]), int(m[4])), {})
        elif line.startswith(".end_amdhsa_kernel"):
            at = None
        elif at is not None and line.startswith(".amdhsa_"):
            key, value = line.split(None, 1)
            at[key[len(".amdhsa_"):]] = value
    return found


def test_as_many_workgroups_on_a_compute_unit_as_the_launch_rules_count_on():
    """512 registers for the wavefronts of a SIMD, given out by 8; 160 KB of LDS for the workgroups of a compute unit."""
    kernels = _kernels()
    for dtype in ("bf16", "f16"):
        forms = {k[1:] for k in kernels if k[0] == dtype}
        assert forms >= {(64, 4, m) for m in range(9)} | {(128, 4, m) for m in range(6)} | {(128, 8, m) for m in (0, 1, 3, 4, 5)}
    for (dtype, d, waves, form), k in kernels.items():
        by_registers = 512 // (-(-int(k["next_free_vgpr"]) // 8) * 8) * 4 // waves
        by_lds = 160 * 1024 // int(k["group_segment_fixed_size"])
        want = 3 if (d, waves) == (64, 4) and form in (0, 3, 5) else 8 // waves
        assert by_registers == want and by_lds >= want, (dtype, d, waves, form, k["next_free_vgpr"], k["group_segment_fixed_size"])
        assert int(k["private_segment_fixed_size"]) == 0, ("registers in memory", dtype, d, waves, form)


@pytest.mark.parametrize("source", sorted(p.name for p in _CSRC.iterdir() if p.suffix in (".hip", ".h")))
def test_no_vector_instruction_in_inline_assembly(source):
    """A vector instruction may read what a matrix instruction wrote some wait states later only. The compiler counts them, but does not
    look into inline assembly."""
    text = (_CSRC / source).read_text()
    for m in re.finditer(r"\basm\b(?:\s+volatile)?\s*\(", text):
        code = "".join(re.findall(r'"((?:[^"\\]|\\.)*)"', text[m.end():text.index(";", text.index(")", m.end()))].split(":")[0]))
        assert not re.search(r"(^|[\s;]|\\[nt])v_", code), code
