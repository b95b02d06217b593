"""What the kernels' asm has to say to the compiler, read from the sources, and to keep itself, read from the built library."""
import re
import shutil
import subprocess
from pathlib import Path

import pytest

CSRC = Path(__file__).resolve().parent.parent / "qwen-engine_amd" / "csrc"


def test_statements_that_need_m0_say_so():
    """An asm statement whose instructions use m0 has it among its operands or among what it overwrites: else the compiler may keep a
    value of its own there across the statement."""
    seen = 0
    for path in sorted(CSRC.glob("*")):
        if path.suffix not in (".hip", ".h"):
            continue
        for text in re.findall(r"\basm\b[^;]*", path.read_text()):
            code, _, operands = text.replace("\\\n", "\n").partition(": :")
            if re.search(r"\bm0\b|\blds\b", code):
                seen += 1
                assert re.search(r'"\{?m0\}?"', operands), f"{path.name}: {text}"
    assert seen


def _scalars(text):
    """The numbers of the scalar registers in an operand."""
    out = set()
    for a, b, c in re.findall(r"\bs(?:\[(\d+):(\d+)\]|(\d+)\b)", text):
        out |= set(range(int(a), int(b) + 1)) if a else {int(c)}
    return out


def test_loads_to_shared_memory_wait_for_their_scalar_operands(tmp_path):
    """A buffer load needs five wait states behind a vector instruction that wrote one of its scalar operands.  The compiler puts them
    before its own loads, but not before those that asm brings."""
    from qwen_engine_amd.kernels import build
    objdump = shutil.which("llvm-objdump") or "/opt/rocm/llvm/bin/llvm-objdump"
    if not Path(objdump).exists():
        pytest.skip("no llvm-objdump")
    lib = tmp_path / "lib.so"
    shutil.copy(build.library_path(), lib)
    subprocess.run([objdump, "--offloading", lib.name], cwd=tmp_path, check=True, capture_output=True)
    loads, early = 0, []
    for part in sorted(tmp_path.glob("*gfx950")):
        if b"kernel" not in part.read_bytes():
            continue
        text = subprocess.run([objdump, "-d", "--no-show-raw-insn", "--no-leading-addr", part.name], cwd=tmp_path, check=True,
                              capture_output=True, text=True).stdout
        kernel, before = "", []                            # before: what each of the last instructions wrote, and its wait states
        for line in text.splitlines():
            if line.endswith(">:"):
                kernel, before = line, []
                continue
            op, _, operands = line.split("//")[0].strip().partition(" ")
            states, wrote = 1, set()
            if op == "s_nop":
                states += int(operands, 0)
            elif op.startswith("v_"):
                # (the results come first: a scalar one alone, or behind a vector one)
                first = operands.split(", ")
                wrote = _scalars(first[0]) | (_scalars(first[1]) if re.match(r"v_(add|sub|subrev|addc|subb|subbrev)_co_|v_div_scale|v_mad_[iu]64", op) else set())
            elif op.startswith("buffer_load") and operands.endswith(" lds"):
                loads += 1
                waited = 0
                for s, w in reversed(before):
                    if waited >= 5:
                        break
                    if w & _scalars(operands):
                        early.append((kernel, line.strip()))
                        break
                    waited += s
            before = before[-7:] + [(states, wrote)]
    assert loads and not early, early[:4]
