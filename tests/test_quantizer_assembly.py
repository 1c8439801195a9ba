"""What the fused quantizer's generated gfx950 code has to show and no run on a GPU shows reliably (CPU test: the file is
compiled to assembly with the library's own flags and read).

A permlane swap must not read a vector register in the two wait states after a vector instruction wrote it, and neither
must an operand read through DPP.  The compiler keeps that distance for the instructions it knows and not for inline assembly.

Where lanes of a wave hand each other values through LDS, the source has to demand the order of the writes and the reads;
a wave barrier (no instruction, a comment in the assembly) shows that it does."""

import os
import re
import subprocess

import pytest

from gemmlib_amd import build

SOURCE = "blkq4_prepack.hip"
WAIT_STATES = 2


@pytest.fixture(scope="module")
def kernels(tmp_path_factory):
    """kernel symbol -> its instructions (comments are kept: the wave barrier is one)"""
    out = tmp_path_factory.mktemp("asm") / "prepack.s"
    subprocess.run([build.HIPCC, *build.HIP_FLAGS, *build.EXTRA_HIP_FLAGS.get(SOURCE, []), "-I", build.INCLUDE, "-I", build.CSRC,
                    "--cuda-device-only", "-S", os.path.join(build.CSRC, SOURCE), "-o", str(out)], check=True, capture_output=True)
    found, name = {}, None
    for line in out.read_text().splitlines():
        label = re.match(r"(_Z\w+):", line)
        if label:
            name = label.group(1)
            found[name] = []
        elif line.startswith("\t.section") or line.startswith("\t.amdhsa"):
            name = None
        elif name and line.strip():
            found[name].append(line.strip())
    return {k: v for k, v in found.items() if "prepack" in k}


def _registers(operand):
    one = re.fullmatch(r"[-|]*v(\d+)\|?", operand)
    if one:
        return {int(one.group(1))}
    several = re.fullmatch(r"[-|]*v\[(\d+):(\d+)\]\|?", operand)
    return set(range(int(several.group(1)), int(several.group(2)) + 1)) if several else set()


def _too_close(lines):
    """(writer, reader) pairs with fewer than WAIT_STATES wait states between them, in the order of the code"""
    pairs, behind = [], []   # behind: (instruction, registers it writes, wait states it takes), latest last
    for line in lines:
        text = line.split(";")[0].strip()
        if not re.match(r"(v|s|ds|global|buffer|flat|scratch)_", text):
            continue
        mnemonic, _, rest = text.partition(" ")
        operands = [o.strip().split(" ")[0] for o in rest.split(",")]
        swap = re.match(r"v_permlane(16|32)_swap", mnemonic)
        dpp = mnemonic.startswith("v_") and re.search(r"\b(quad_perm|row_\w+|wave_\w+):?", rest)
        if swap or dpp:
            reads = _registers(operands[0]) | _registers(operands[1]) if swap else _registers(operands[1])
            waited = 0
            for writer, written, states in reversed(behind):
                if waited >= WAIT_STATES:
                    break
                if written & reads:
                    pairs.append((writer, text))
                    break
                waited += states
        written = set()
        if mnemonic.startswith("v_"):
            written = _registers(operands[0]) | (_registers(operands[1]) if swap else set())
        behind.append((text, written, int(operands[0], 0) + 1 if mnemonic == "s_nop" else 1))
    return pairs


def test_cross_lane_instructions_keep_their_distance_from_what_they_read(kernels):
    along_n = [k for k in kernels if "rowwise" in k]
    assert len(along_n) == 12 * 2 and len(kernels) == 2 * len(along_n)   # block sizes x zero-points x alignment x types
    for name in along_n:
        assert any("v_permlane32_swap" in line for line in kernels[name]), name
    bad = {name: pairs for name, lines in kernels.items() if (pairs := _too_close(lines))}
    assert not bad, bad


@pytest.mark.parametrize("bs", [16, 32, 64])
def test_values_handed_over_inside_a_wave_are_ordered_by_the_source(kernels, bs):
    """blocks along N: one hand-over of reciprocals and zero-points per block of the tile, ordered on both sides"""
    blocks = {16: 4, 32: 1, 64: 1}[bs]   # of a tile: 64 / 16, 32 / 32 and 64 / 64 columns
    names = [k for k in kernels if f"rowwise_kernelILi{bs}E" in k]
    assert len(names) == 8
    for name in names:
        assert sum("wave barrier" in line for line in kernels[name]) == 2 * blocks, name


def test_the_distance_check_sees_what_it_is_meant_to_see():
    assert _too_close(["v_pk_max_f16 v16, v16, v17", "v_permlane32_swap_b32_e32 v10, v14", "v_permlane32_swap_b32_e32 v11, v16"])
    assert _too_close(["v_add_u32_e32 v1, v2, v3", "s_nop 0", "v_mov_b32_dpp v4, v1 row_ror:8 row_mask:0xf bank_mask:0xf"])
    assert not _too_close(["v_add_u32_e32 v1, v2, v3", "s_nop 1", "v_mov_b32_dpp v4, v1 row_ror:8 row_mask:0xf bank_mask:0xf"])
    assert not _too_close(["v_add_u32_e32 v1, v2, v3", "v_mov_b32_e32 v4, v1"])
