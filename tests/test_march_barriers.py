"""Block barriers of the column marches: a barrier must be reached by every wave of the block, so none
may stand in a branch, nor in a function that is called from one (the two-threads-per-column march
branches between its waves)."""
import os
import re

import pytest

from astaroth_amd.build import CSRC


def blocks_around(text, pos):
    """Headers (the text before each opening brace, back to the last ; { or }) of the blocks that
    contain `pos`, innermost first."""
    headers, depth = [], 0
    for i in range(pos - 1, -1, -1):
        if text[i] == "}":
            depth += 1
        elif text[i] == "{":
            if depth == 0:
                start = max(text.rfind(c, 0, i) for c in ";{}")
                headers.append(text[start + 1:i].strip())
            else:
                depth -= 1
    return headers


def in_branch(text, pos):
    """Whether the statement at `pos` runs under an if or else of its function."""
    before = text[:pos].rstrip()
    if re.search(r"\belse$", before) or (before.endswith(")") and re.search(r"\bif\s*\([^;{}]*\)$", before)):
        return True
    for header in blocks_around(text, pos):
        if re.search(r"\b(if|else|switch)\b", header.split("\n")[-1]):
            return True
        if re.search(r"__device__", header):
            return False
    return False


@pytest.mark.parametrize("name", ["solve_ring.h", "solve_pair.h"])
def test_barriers_stand_outside_branches(name):
    with open(os.path.join(CSRC, name)) as f:
        text = re.sub(r"//[^\n]*", "", f.read())
    barriers = [m.start() for m in re.finditer(r"__syncthreads\(\)", text)]
    assert barriers
    functions = set()
    for pos in barriers:
        assert not in_branch(text, pos), text[max(0, pos - 200):pos + 20]
        for header in blocks_around(text, pos):
            if "__device__" in header:
                functions.add(re.search(r"(\w+)\s*\([^()]*\)\s*(const)?$", header).group(1))
                break
    assert functions
    for fn in functions:
        calls = [m.start() for m in re.finditer(r"(?<![\w~])%s\s*(<\w+>)?\(" % fn, text)]
        for pos in calls:
            assert not in_branch(text, pos), (fn, text[max(0, pos - 120):pos + 60])
