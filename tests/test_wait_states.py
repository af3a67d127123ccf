"""Wait states around the direct-to-LDS loads that are written in assembly, where the compiler does not
insert them: a vector-memory instruction that reads an SGPR written by a VALU instruction needs five
wait states between the two."""

from __future__ import annotations

import re
import shutil
import subprocess
from pathlib import Path

import pytest

REPO_ROOT = Path(__file__).resolve().parent.parent
CSRC = REPO_ROOT / "llm-serving-engine_amd" / "csrc"
NEEDED = 5
VMEM = re.compile(r"(buffer|global|flat|scratch)_")


def _states(op: str, args: str) -> int:
    return int(args, 0) + 1 if op == "s_nop" else 1


def test_the_scalar_base_loads_wait_by_themselves():
    """Whatever the compiler puts before the assembly block, its own instructions make up the wait."""
    source = (CSRC / "attn_tile.hip").read_text()
    block = source[source.index("void dma4_saddr"):]
    states = 0
    for op, args in re.findall(r'"(\w+) ?([^"\\]*)(?:\\n\\t)?"', block):
        if VMEM.match(op):
            break
        states += _states(op, args)
    assert states >= NEEDED


def _registers(operand: str) -> set[int]:
    m = re.fullmatch(r"s\[(\d+):(\d+)\]", operand)
    if m:
        return set(range(int(m[1]), int(m[2]) + 1))
    m = re.fullmatch(r"s(\d+)", operand)
    return {int(m[1])} if m else set()


def _early_reads(listing: str) -> list[str]:
    """Vector-memory instructions that read an SGPR fewer than NEEDED wait states after a VALU
    instruction wrote it, in the order of the listing."""
    found, since = [], {}  # SGPR -> wait states since a VALU instruction wrote it
    for line in listing.splitlines():
        m = re.match(r"\s+([a-z]\w+)\s*([^/]*)", line)
        if not m:
            continue
        op, operands = m[1], [o.split()[0] for o in re.split(r",(?![^\[]*\])", m[2]) if o.strip()]
        if VMEM.match(op):
            if any(since.get(r, NEEDED) < NEEDED for o in operands for r in _registers(o)):
                found.append(line.strip())
        states = _states(op, operands[0] if operands else "0")
        since = {r: n + states for r, n in since.items() if n + states < NEEDED}
        if op.startswith(("v_readlane", "v_readfirstlane", "v_cmp")) and operands:
            since.update(dict.fromkeys(_registers(operands[0]), 0))
    return found


def test_the_check_sees_an_early_read():
    early = "\tv_readlane_b32 s5, v1, 3\n\ts_nop 3\n\tglobal_load_lds_dwordx4 v2, s[4:5]\n"
    assert len(_early_reads(early)) == 1
    assert not _early_reads(early.replace("s_nop 3", "s_nop 4"))


def test_no_kernel_reads_a_scalar_too_early(pkg, tmp_path):
    objdump = shutil.which("llvm-objdump") or "/opt/rocm/lib/llvm/bin/llvm-objdump"
    if not Path(objdump).exists():
        pytest.skip("needs llvm-objdump")
    lib = tmp_path / "lib.so"
    shutil.copy(pkg.LIB_PATH, lib)
    subprocess.run([objdump, "--offloading", lib.name], cwd=tmp_path, check=True,
                   capture_output=True)
    objects = sorted(tmp_path.glob("*gfx950"))
    assert objects
    loads = 0
    for obj in objects:
        listing = subprocess.run([objdump, "-d", "--no-show-raw-insn", obj.name], cwd=tmp_path,
                                 check=True, capture_output=True, text=True).stdout
        loads += listing.count(" lds")
        assert not _early_reads(listing), obj.name
    assert loads > 0
