"""Source check of the kernels' out-of-range buffer reads.

A read that is not to happen is given an offset past its descriptor's byte
count, and the hardware returns zeros for it. That holds for the lane offset
(the second operand of a raw buffer load): the range check compares it with
the byte count less the scalar offset (the operand after it), so an
out-of-range marker in the scalar offset makes that difference wrap and may
let the read through, 2 GiB past the buffer. This test reads every raw buffer
load in csrc/ and fails where the scalar offset holds such a marker, directly
or through a local variable made from one.
"""
import re
from pathlib import Path

import pytest

CSRC = Path(__file__).resolve().parent.parent / "nemotron-webgpu-decode_amd" / "csrc"
# (after an & the number is a mask: of a float's sign, of a nibble's place)
MARKER = re.compile(r"(?<!& )\b(kNoRead|oob|0x80000000u?|0x7FFFFFFFu?)\b", re.I)
LOADS = re.compile(r"__builtin_amdgcn_raw_(ptr_)?buffer_load_(\w+)\s*\(")


def _operands(text: str, at: int) -> list:
    """The comma-separated operands of the call whose '(' is at `at`."""
    out, depth, start = [], 0, at + 1
    for i in range(at, len(text)):
        ch = text[i]
        if ch in "([{":
            depth += 1
        elif ch in ")]}":
            depth -= 1
            if depth == 0:
                return out + [text[start:i].strip()]
        elif ch == "," and depth == 1:
            out.append(text[start:i].strip())
            start = i + 1
    raise AssertionError("unbalanced call")


def _violations(text: str):
    text = re.sub(r"//[^\n]*", "", text)
    made = {m.group(1) for m in re.finditer(r"\b(\w+)\s*=\s*([^;]*);", text) if MARKER.search(m.group(2))}
    found, checked = [], 0
    for m in LOADS.finditer(text):
        ops = _operands(text, m.end() - 1)
        # (rsrc, lane, scalar, aux); to LDS: (rsrc, lds, size, lane, scalar, imm, aux)
        scalar = ops[4] if m.group(2) == "lds" else ops[2]
        checked += 1
        if MARKER.search(scalar) or any(w in made for w in re.findall(r"\b[A-Za-z_]\w*", scalar)):
            found.append(" ".join(scalar.split()))
    return found, checked


def test_checker_flags_a_marker_in_the_scalar_offset():
    ok = "x = __builtin_amdgcn_raw_buffer_load_b32(r, in ? f(a, b) : kNoRead, c * 4, 0);"
    direct = "x = __builtin_amdgcn_raw_buffer_load_b32(r, lane * 4, in ? f(a, b) : kNoRead, 0);"
    named = "const int off = in ? 0 : kNoRead; __builtin_amdgcn_raw_ptr_buffer_load_lds(r, d, 16, l, n | off, 0, 0);"
    assert _violations(ok) == ([], 1)
    assert len(_violations(direct)[0]) == 1 and len(_violations(named)[0]) == 1


@pytest.mark.parametrize("unit", sorted(p.name for p in CSRC.glob("*") if p.suffix in (".h", ".hip")))
def test_scalar_offsets_hold_no_out_of_range_marker(unit):
    found, _ = _violations((CSRC / unit).read_text())
    assert not found, found
