"""The state scans' requests (csrc/gdn_fwd.hip, gdn_bwd.hip) against the rule of ScanBlocks in
csrc/gdn_common.hpp: a step past the last is given the buffer's size as its scalar offset, which the
range check of a raw buffer (lane offset >= size - scalar offset) turns away lane by lane.  Anything
added to that scalar would make the difference wrap around, so what a lane adds belongs in its own
offset."""

import re
from pathlib import Path

import pytest

CSRC = Path(__file__).resolve().parents[1] / "cq-pretrain_amd" / "csrc"


def _arguments(text, at):
    """The top-level arguments of the call whose opening parenthesis is text[at]."""
    depth, start, args = 0, at + 1, []
    for i in range(at, len(text)):
        c = text[i]
        depth += c in "([{"
        depth -= c in ")]}"
        if depth == 0 or (depth == 1 and c == ","):
            args.append(" ".join(text[start:i].split()))
            start = i + 1
        if depth == 0:
            return args
    raise AssertionError("unbalanced call")


def _requests(name):
    """(buffer, scalar offset) of every buffer access of the scan kernel's source with one."""
    text = re.sub(r"//.*", "", (CSRC / name).read_text())
    out = []
    for m in re.finditer(r"\bbuf_(?:ld|st)\w*\s*(?:<[^<>()]*>)?\s*\(", text):
        args = _arguments(text, m.end() - 1)
        if ".offset(" in " ".join(args):
            out.append(args)
    return out


@pytest.mark.parametrize("name,least", [("gdn_fwd.hip", 4), ("gdn_bwd.hip", 6)])
def test_scalar_offsets_are_the_blocks_alone(name, least):
    calls = _requests(name)
    assert len(calls) >= least, calls
    for args in calls:
        scalar = args[2] if len(args) > 2 and ".offset(" in args[2] else None
        if scalar is None:  # a 16-byte store has no scalar offset: its lane offset holds the block's
            assert len(args) == 3 and re.fullmatch(r"\w+ \+ \w+\.offset\(\w+\)", args[1]), args
            continue
        assert re.fullmatch(r"\w+\.offset\(\w+\)", scalar), args
        assert ".offset(" not in args[1], args
