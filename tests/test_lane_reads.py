"""v_readlane of another lane's register is defined only while that lane takes part: inside a branch
that some lanes do not take, a value that the compiler moved or reloaded there exists for the taking
lanes alone. The kernels therefore read lanes before a branch on the lane, never inside it. Checked
on the sources: no lane read, and no call of a function or lambda that holds one, in the body of an
`if` on the lane or on a lane mask, or after an early `continue` / `return` of such an `if`."""
import glob
import os
import re

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
SOURCES = sorted(glob.glob(os.path.join(ROOT, "masterthesislucas_amd", "csrc", "*.h*")))
ON_LANE = re.compile(r"inverse_ballot|\blane\b")


def _matching(s, i, a, b):
    """Index after the bracket that closes the one at s[i]."""
    depth = 0
    for j in range(i, len(s)):
        depth += (s[j] == a) - (s[j] == b)
        if depth == 0:
            return j + 1
    raise ValueError("unbalanced source")


def _block_end(s, i):
    """End of the block that holds position i."""
    depth = 0
    for j in range(i, len(s)):
        depth += (s[j] == "{") - (s[j] == "}")
        if depth < 0:
            return j
    return len(s)


def _statement_end(s, i):
    while s[i].isspace():
        i += 1
    if s[i] == "{":
        return _matching(s, i, "{", "}")
    m = re.compile(r"(if constexpr|if|for|while)\s*\(").match(s, i)
    if m:
        return _statement_end(s, _matching(s, m.end() - 1, "(", ")"))
    return s.index(";", i) + 1


def _readers(s):
    """Names of what holds a lane read, directly or through a call."""
    bodies = {}
    for m in re.finditer(r"\bauto (\w+) = \[&\]\s*\(|\b(\w+)\s*\(", s):
        name = m.group(1) or m.group(2)
        if name in ("if", "for", "while", "switch", "constexpr"):
            continue
        end = _matching(s, m.end() - 1, "(", ")")
        head = re.compile(r"\s*(const\s*)?\{").match(s, end)
        if head:
            bodies[name] = bodies.get(name, "") + s[head.end() - 1:_matching(s, head.end() - 1, "{", "}")]
    found = {"__builtin_amdgcn_readlane"}
    while True:
        call = re.compile(r"\b(%s)\s*\(" % "|".join(found))
        # (a kernel or a function that calls a lambda of its own holds it as a whole: not a call of it)
        more = {n for n, b in bodies.items() if n not in found and call.search(b)}
        if not more:
            return call
        found |= more


def masked_lane_reads(text):
    s = re.sub(r"//[^\n]*|/\*.*?\*/", lambda m: re.sub(r"[^\n]", " ", m.group()), text, flags=re.S)
    call = _readers(s)
    hits = []
    for m in re.finditer(r"\bif\s*(constexpr\s*)?\(", s):
        end = _matching(s, m.end() - 1, "(", ")")
        if not ON_LANE.search(s[m.end():end]):
            continue
        stop = _statement_end(s, end)
        if re.match(r"\s*\{?\s*(continue|return)\b", s[end:stop]):
            stop = _block_end(s, stop)
        h = call.search(s, end, stop)
        if h:
            hits.append((s.count("\n", 0, h.start()) + 1, h.group()))
    return hits


@pytest.mark.parametrize("path", SOURCES, ids=os.path.basename)
def test_lanes_are_read_before_the_branch(path):
    with open(path) as f:
        assert masked_lane_reads(f.read()) == []


def test_the_check_sees_them():
    read = "uint32_t lane_read(uint32_t v, uint32_t l) { return __builtin_amdgcn_readlane(v, l); }\n"
    masked = ["if (lane > o) { x = lane_read(v, e); }", "if (lane > o) x = lane_read(v, e);",
              "auto f = [&](int k) { return lane_read(v, k); };\nif (on(inverse_ballot(m))) f(1);",
              "if (!inverse_ballot(m)) continue;\nx = lane_read(v, e);"]
    fine = ["y = lane_read(v, e);\nif (lane > o) x = y;", "if (n > o) x = lane_read(v, e);"]
    for body in masked + fine:
        got = masked_lane_reads(read + "void k() { for (;;) { " + body + " } }")
        assert bool(got) == (body in masked), body
