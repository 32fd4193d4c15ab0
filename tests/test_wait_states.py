"""Wait states that the hardware asks of software, in the library as built.

The compiler keeps them between its own instructions but does not look inside ``asm`` statements. The check reads the
disassembly of ``libjigsaw_hip.so`` (AMD assembly of this repository's sources, all of it).
"""

from __future__ import annotations

import re
import subprocess
from pathlib import Path

import pytest

from jigsaw_amd import _lib

OBJDUMP = Path("/opt/rocm/llvm/bin/llvm-objdump")
_REGS = re.compile(r"\bs(\d+)\b|\bs\[(\d+):(\d+)\]")


def _scalars(text: str) -> set:
    """Scalar registers named in the operands."""
    return {r for one, lo, hi in _REGS.findall(text) for r in (range(int(one), int(one) + 1) if one else range(int(lo), int(hi) + 1))}


def _m0_too_soon(lines) -> list:
    """Transfers to LDS less than one wait state behind a scalar write of the M0 they read."""
    return [f"{a} / {b}" for a, b in zip(lines, lines[1:]) if b.startswith("global_load_lds") and a.startswith("s_") and a.split()[1:2] == ["m0,"]]


_RULES = {"m0": _m0_too_soon}


@pytest.fixture(scope="module")
def code(tmp_path_factory):
    """Instructions of every device code object, in order."""
    if not OBJDUMP.exists():
        pytest.skip("no llvm-objdump")
    lib = Path(_lib.lib_path())
    if not lib.exists():
        pytest.skip("the library is not built")
    where = tmp_path_factory.mktemp("code")
    (where / lib.name).symlink_to(lib.resolve())
    subprocess.run([OBJDUMP, "--offloading", lib.name], cwd=where, check=True, capture_output=True)
    objects = sorted(where.glob("*gfx950*"))
    assert objects
    lines = []
    for o in objects:
        out = subprocess.run([OBJDUMP, "-d", "--no-leading-addr", "--no-show-raw-insn", o], check=True, capture_output=True, text=True).stdout
        lines += [ln.split("//")[0].strip() for ln in out.splitlines() if ln.startswith("\t")]
    assert any(ln.startswith("global_load_lds") for ln in lines)
    return lines


@pytest.mark.parametrize("rule", _RULES)
def test_asm_statements_keep_the_wait_states(rule, code):
    found = _RULES[rule](code)
    assert not found, f"{len(found)}, the first: {found[:3]}"
