"""The 2D push's LDS counters between its barriers: what a pass stores, adds to
and reads without an order between the threads never shares a stretch of code
between two barriers.  (A store of zero beside the reads of the list of moves
that leave the window could hide a wave's share of them.)"""
import os
import re

import pytest

SRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                   "tristan-mp-pu-master_densdecomp_amd", "csrc", "push2d.hip")


def _stretches():
    """the code of the pass loop between barriers; what follows the last
    barrier runs beside what precedes the next pass's first"""
    s = re.sub(r"//.*", "", open(SRC).read())
    a = s.index("for (int pass = 0;")
    at = s.index("{", a)
    depth, end = 0, at
    for end in range(at, len(s)):
        depth += {"{": 1, "}": -1}.get(s[end], 0)
        if depth == 0:
            break
    parts = s[at:end].split("__syncthreads();")
    assert len(parts) == 5, "the barriers of a pass"
    return [parts[-1] + parts[0]] + parts[1:-1]


@pytest.mark.parametrize("name,element", [("nx_list", r"\*nx_list"), ("nitem", r"\*nitem"), ("cnt", r"\bcnt\[[^]]*\]"),
                                          ("start", r"\bstart\[[^]]*\]")])
def test_counters_change_between_barriers(name, element):
    uses = []
    for code in _stretches():
        kinds = set()
        if re.search(element + r"\s*=[^=]", code):
            kinds.add("store")
        if re.search(element + r"(?!\s*=[^=])", code):
            kinds.add("read")
        if re.search(r"atomicAdd\(" + name + r"\b", code):
            kinds.add("add")
        uses.append(kinds)
    assert all(len(k) <= 1 for k in uses), uses
    assert {"store", "read"} <= set().union(*uses)
