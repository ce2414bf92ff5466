"""How the two kinds of waves of a recurrence (walk) workgroup leave together when a wait gives up, read from the kernels'
sources: the word that says so may not be written between two barriers between which any wave reads it.  Where it is, one
wave can see it and return while another misses it, goes on and waits for the first one's arrival, a wait that has no limit."""
import os
import re

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "ttt-tk_amd", "csrc")


def _block(text, start):
    """(inside of the braces that open at or after `start`, index behind the closing one)"""
    i = text.index("{", start)
    depth = 0
    for j in range(i, len(text)):
        depth += {"{": 1, "}": -1}.get(text[j], 0)
        if depth == 0:
            return text[i + 1:j], j + 1
    raise ValueError("unbalanced braces")


def _inline(text):
    """`text` with its named lambdas put in the place of their calls."""
    bodies = {}
    while (m := re.search(r"\bauto (\w+) = \[&\]\([^)]*\) ", text)) is not None:
        body, end = _block(text, m.end())
        bodies[m.group(1)] = body
        text = text[:m.start()] + text[end:]
    bodies.pop("flag", None)
    for _ in range(4):
        for name, body in bodies.items():
            text = re.sub(r"\b" + name + r"\(", lambda _m: body + "(", text)
    return text


EVENTS = re.compile(r"(?P<B>__syncthreads\(\))|(?P<W>s_flag\[0\] = 1|\*s_flag = 1)|(?P<R>\bflag\(0?\))")


def _intervals(text, loop):
    """Events between barriers of prologue, two passes of the loop and epilogue, one string per interval."""
    at = text.index(loop)
    body, end = _block(text, at)
    seq = [m.lastgroup for part in (text[:at], body, body, text[end:]) for m in EVENTS.finditer(part)]
    return "".join(seq).split("B")


@pytest.mark.parametrize("source,function,loop", [
    ("ttt_mlp_bwd_wide.hip", "bwd_wide_walk", "for (int k = p.K - 1; k >= 0; k--)"),
    ("ttt_mlp_fwd_wide.hip", "fwd_wide_recurrence", "for (int mb = 0; mb < p.NC; mb++)")])
def test_leaving_is_decided_between_barriers_by_all_waves_alike(source, function, loop):
    text = re.sub(r"//[^\n]*", "", open(os.path.join(CSRC, source)).read())
    body, _ = _block(text, text.index("TTT_DEV void " + function))
    at = re.search(r"if \((w < 4|compute|v < WD_NCOMP|w < WD_NCOMP)\) ", body)
    compute, end = _block(body, at.end())
    kinds = [_intervals(_inline(kind), loop) for kind in (compute, body[end:])]
    assert len(kinds[0]) == len(kinds[1]) > 7, "both kinds of waves pass the same barriers"
    assert any("W" in x for x in kinds[1]) and any("R" in x for x in kinds[0])
    for i, (a, b) in enumerate(zip(*kinds)):
        assert not ("W" in a + b and "R" in a + b), f"interval {i}: the word is written while it is read ({a!r}, {b!r})"


def test_the_count_of_gathered_sums_orders_what_it_counts():
    """The compute waves overwrite block 0's partial sums once four helpers have counted up: a release before the count, an
    acquire behind the wait (in the forward, the shares of b2 the same way)."""
    text = re.sub(r"//[^\n]*", "", open(os.path.join(CSRC, "ttt_mlp_bwd_wide.hip")).read())
    assert re.search(r'fence\(__ATOMIC_RELEASE, "workgroup", "local"\);\s*if \(lane == 0\) __hip_atomic_fetch_add\(s_flag \+ 1', text)
    assert re.search(r'while \(flag\(1\) < 4 \* \(n \+ 1\)\)[^;]*;\s*__builtin_amdgcn_fence\(__ATOMIC_ACQUIRE, "workgroup", "local"\)', text)
    text = open(os.path.join(CSRC, "ttt_mlp_fwd_wide.hip")).read()
    assert "__hip_atomic_fetch_add(s_flag + 1, 1, __ATOMIC_RELEASE" in text
    assert re.search(r'while \(__hip_atomic_load\(s_flag \+ 1[^;]*;\s*__builtin_amdgcn_fence\(__ATOMIC_ACQUIRE, "workgroup"\)', text)
