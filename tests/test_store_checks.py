"""Source checks of the launchers and of the bounds-checked build.

In the bounds-checked build the kernels of csrc/nwd_q4_rows.hip compare every
store into an output, a cache or the workspace with its buffer (in_bounds, or
in_scratch for the workspace).

Every statement of its device code that stores through one of those pointers
must hold such a check, or follow one that leaves (return, continue) directly
in the same block.
"""
import re
from pathlib import Path

SRC = (Path(__file__).resolve().parent.parent / "nemotron-webgpu-decode_amd" / "csrc" / "nwd_q4_rows.hip")
CHECK = re.compile(r"\bin_(bounds|scratch)\(")
# stores through the pointers of the kernels' arguments
STORES = re.compile(
    r"(p\.records\[[^;=]*\]|p\.y\[[^;=]*\]|\*y|\bo\[\d+\]|\bfactor\[[^;=]*\]|\bwide_best\[[^;=]*\]|\*wide_tickets"
    r"|\*at|_cache\)\[[^;=]*\]|p\.q_out\)\[[^;=]*\])\s*=[^=]")


def _unchecked(text: str):
    code = re.sub(r"//[^\n]*", "", text)
    bad, seen = [], 0
    for m in STORES.finditer(code):
        seen += 1
        # back over the block's statements up to its check, or its opening
        depth, i = 0, m.start()
        while i > 0:
            i -= 1
            if code[i] == "}":
                depth += 1
            elif code[i] == "{":
                if depth == 0:
                    break
                depth -= 1
        if not CHECK.search(code[i:m.start()]):
            bad.append(" ".join(m.group(0).split()))
    return bad, seen


def test_checker_flags_a_store_without_a_check():
    ok = "{ if (!in_bounds(at, 1, n, s)) return; p.y[at] = v; }"
    assert _unchecked(ok) == ([], 1)
    assert _unchecked("{ if (in_bounds(at, 1, n, s)) f(); } { p.y[at] = v; }") == (["p.y[at] ="], 1)


def test_every_store_is_checked():
    bad, seen = _unchecked(SRC.read_text())
    assert seen >= 11, f"only {seen} stores found"
    assert not bad, bad


def test_lds_limits_are_raised_once_per_device():
    """hipFuncSetAttribute (a runtime call of its own, which a call of few
    microseconds shows) is not part of every launch: a per-device bit goes
    before it in its function."""
    seen = 0
    for path in sorted(SRC.parent.glob("*")):
        if path.suffix not in (".h", ".hip"):
            continue
        for block in re.split(r"\n}", path.read_text()):  # top-level functions
            for m in re.finditer(r"hipFuncSetAttribute\(", block):
                seen += 1
                assert "attr_set.load()" in block[:m.start()], path.name
    assert seen >= 4
