"""CPU checks of the kernels' source text.  Requests that may start inside an
operand and reach past its end: the buffer resource's range check compares the
vector offset (and the instruction's constant) with the operand's size, and
the scalar offset is documented to be outside of it, so every request of these
sources carries its whole offset in the vector part.  And inline assembly
names the registers it writes."""
import os
import re

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "infer_amd", "csrc")


def arguments(text, start):
    """The top-level arguments of the call whose '(' is at start."""
    depth, args, cur = 0, [], ""
    for c in text[start:]:
        if c in "([{":
            depth += 1
            if depth == 1:
                continue
        elif c in ")]}":
            depth -= 1
            if depth == 0:
                return [a.strip() for a in args + [cur]]
        if c == "," and depth == 1:
            args.append(cur)
            cur = ""
        else:
            cur += c
    raise AssertionError("unbalanced call")


@pytest.mark.parametrize("name", ["iq_gemmw.hip", "iq_quant.hip"])
def test_requests_are_range_checked_whole(name):
    with open(os.path.join(CSRC, name)) as f:
        text = re.sub(r"//[^\n]*", "", f.read())
    calls = list(re.finditer(r"__builtin_amdgcn_raw_(?:ptr_)?buffer_load_\w+\(", text))
    for m in calls:
        args = arguments(text, m.end() - 1)
        assert len(args) == 4 and args[2] == "0", f"{name}: scalar offset {args[2]!r} in {args}"
    asm = re.findall(r"buffer_load_\w+ [^\"\\]*", text)
    asm = [a for a in asm if "%" in a]
    for a in asm:
        assert re.match(r"buffer_load_\w+ %\d+, %\d+, 0 offen", a), f"{name}: scalar offset in {a!r}"
    assert calls or asm


def test_asm_that_writes_m0_says_so():
    for name in sorted(os.listdir(CSRC)):
        if not name.endswith((".hip", ".h")):
            continue
        with open(os.path.join(CSRC, name)) as f:
            text = re.sub(r"//[^\n]*", "", f.read())
        for m in re.finditer(r"asm(?:\s+volatile)?\s*\(", text):
            call = text[m.end() - 1:text.index(";", m.end())]
            if re.search(r"\bm0,", call):
                assert '"m0"' in call, f"{name}: {call}"
