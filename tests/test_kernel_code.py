"""The machine code of the built library, read on the CPU: what the tile engine's asm
statements and its speed rest on and what a change of the compiler or of the code around
them could take away without any result changing at first."""

import os
import re
import shutil
import struct
import subprocess

import pytest

from turbo_dllm_amd import _lib
from turbo_dllm_amd.build import find_hipcc

DIRECT = "MfmaDirect4Engine"


def _tool(name):
    beside = os.path.join(os.path.dirname(os.path.realpath(find_hipcc())), "..", "llvm", "bin", name)
    return beside if os.path.exists(beside) else shutil.which(name) or f"/opt/rocm/llvm/bin/{name}"


@pytest.fixture(scope="module")
def code_objects(tmp_path_factory):
    """The gfx950 code objects of the library: one per compilation unit."""
    _lib.library()
    data = _lib.LIBRARY_PATH.read_bytes()
    folder = tmp_path_factory.mktemp("code")
    paths, at = [], 0
    while (start := data.find(b"__CLANG_OFFLOAD_BUNDLE__", at)) >= 0:
        entries, = struct.unpack_from("<Q", data, start + 24)
        cursor = start + 32
        for _ in range(entries):
            offset, size, length = struct.unpack_from("<QQQ", data, cursor)
            name = data[cursor + 24:cursor + 24 + length]
            cursor += 24 + length
            if b"gfx950" in name:
                paths.append(folder / f"{len(paths)}.elf")
                paths[-1].write_bytes(data[start + offset:start + offset + size])
        at = start + 24
    assert paths, "no gfx950 code in the library"
    return paths


@pytest.fixture(scope="module")
def kernels(code_objects):
    """name -> (metadata, instructions) of every kernel of the direct engine."""
    found = {}
    for path in code_objects:
        notes = subprocess.run([_tool("llvm-readelf"), "--notes", path], capture_output=True,
                               text=True, check=True).stdout
        if DIRECT not in notes:
            continue
        meta = {}
        for block in notes.split("- .agpr_count")[1:]:
            name = re.search(r"\.name: +(\S+)", block)[1]
            meta[name] = {key: int(value) for key, value in
                          re.findall(r"\.(private_segment_fixed_size|vgpr_spill_count): +(\d+)", block)}
        text = subprocess.run([_tool("llvm-objdump"), "-d", "--no-show-raw-insn", path],
                              capture_output=True, text=True, check=True).stdout
        name = None
        for line in text.splitlines():
            if (head := re.match(r"[0-9a-f]+ <(\S+)>:", line)):
                name = head[1]
                found[name] = (meta[name], []) if name in meta and DIRECT in name else None
            elif name and found.get(name) and line.startswith("\t"):
                found[name][1].append(line.split("//")[0].strip())
    found = {name: value for name, value in found.items() if value}
    assert len(found) > 20
    return found


def test_forward_statistics_keep_their_running_pairs_in_registers(kernels):
    """A pair in scratch memory is a round trip per tile and column (5 us a tile)."""
    seen = 0
    for name, (meta, _) in kernels.items():
        if "lce_forward_stats_kernel" in name and name.split("EEvNS")[0].endswith("ELb0E"):
            seen += 1
            assert meta == {"private_segment_fixed_size": 0, "vgpr_spill_count": 0}, name
    assert seen == 8       # bf16 and f16, with and without soft cap and bias


def test_main_loops_wait_for_no_more_than_the_tile_they_need(kernels):
    """A K step waits once for its tile (all loads but the youngest).  A wait of the
    compiler's own in there, for a load of the code around the loop, waits for the loads of
    the tile after it as well."""
    loops = 0
    for name, (_, code) in kernels.items():
        for at, line in enumerate(code):
            if not line.startswith("s_cbranch") or at < 150:
                continue
            # a loop of one K step: the branch goes back over 128 MFMAs and no other branch
            body = []
            for back in range(at - 1, max(at - 400, 0), -1):
                if code[back].startswith(("s_cbranch", "s_branch", "s_endpgm")):
                    break
                body.append(code[back])
            target = int(line.split()[1])
            if target < 0x8000 or sum(b.startswith("v_mfma") for b in body) != 128:
                continue
            loops += 1
            waits = [b for b in body if b.startswith("s_waitcnt") and "vmcnt" in b]
            assert waits == ["s_waitcnt vmcnt(1)"], (name, waits)
    assert loops >= len(kernels) // 2


def _registers(operand):
    """v5, v[4:7], a[0:3] -> {("v", 5)} ..."""
    match = re.fullmatch(r"([va])(?:(\d+)|\[(\d+):(\d+)\])", operand.strip())
    if not match:
        return frozenset()
    first = int(match[2] or match[3])
    return frozenset((match[1], r) for r in range(first, int(match[4] or first) + 1))


def _operands(line):
    return [_registers(part) for part in line.partition(" ")[2].split(",")]


def _issued(line):
    """Wait states an instruction stands for (a 16x16x32 MFMA holds its pipe for four)."""
    return int(line.split()[1]) + 1 if line.startswith("s_nop") else 4 if line.startswith("v_mfma") else 1


def test_wait_states_around_the_asm_matrix_instructions(kernels):
    """The compiler adds no wait states for instructions in asm statements: an MFMA must not
    follow a vector instruction that writes one of its operands by less than two of them,
    and its result must not be read by another kind of instruction for 19."""
    checked = 0
    for name, (_, code) in kernels.items():
        parsed = [_operands(line) for line in code]
        for at, line in enumerate(code):
            matrix = line.startswith("v_mfma")
            stores = not line.startswith("v_")
            sources = frozenset().union(*parsed[at][0 if stores else 1:])
            if not matrix:
                sources = frozenset(r for r in sources if r[0] == "a")
            if not sources:
                continue
            checked += 1
            waited, back = 0, at - 1
            while back >= 0 and waited < (2 if matrix else 19):
                before = code[back]
                if before.startswith("v_mfma" if not matrix else "v_") and before.startswith("v_mfma") != matrix:
                    assert not parsed[back][0] & sources, (name, before, line)
                waited += _issued(before)
                back -= 1
    assert checked > 100 * len(kernels)
