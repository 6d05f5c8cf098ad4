"""Order of the LDS words that the panel chain's waves share (bta_flow.hip).

The chain (flow_chain with flow_wait2) passes three results between its waves
through `ok_sh`.  A word that all waves read may be written again only after a
barrier that follows the read: otherwise a wave that reads late sees the next
value, takes another branch than the rest and leaves the barriers out of step.
The loop over the columns is read from the source as a list of accesses and
barriers, with the wait taken and not taken, and run through twice."""
import itertools
import re
from pathlib import Path

SRC = Path(__file__).resolve().parents[1] / "pyinla_amd" / "csrc" / "bta_flow.hip"


def _body(text, name):
    at = re.search(r"__forceinline__ \w+ " + name + r"\(", text).end()
    at = text.index("{", at)
    depth, end = 0, at
    for end in range(at, len(text)):
        depth += {"{": 1, "}": -1}.get(text[end], 0)
        if depth == 0:
            break
    return re.sub(r"//[^\n]*", "", text[at:end])


def _loop(body):
    at = body.index("for (int k = 0; k + 1 < nT; ++k)")
    at = body.index("{", at)
    depth = 0
    for end in range(at, len(body)):
        depth += {"{": 1, "}": -1}.get(body[end], 0)
        if depth == 0:
            return body[at:end]
    raise AssertionError("unbalanced loop")


def _events(body, wait):
    """('B',), ('R', word) and ('W', word) in source order."""
    word = r"(?:ok_sh\[(?P<w>\d)\]|\*ok_sh)"
    pat = re.compile(r"(?P<bar>lds_barrier\(\)|__syncthreads\(\)|flow_publish\()|(?P<wait>flow_wait2\()"
                     r"|(?P<add>atomicAdd\(&ok_sh\[(?P<aw>\d)\])|" + word + r"(?P<write>\s*=[^=])?")
    out = []
    for m in pat.finditer(body):
        if m.group("bar"):
            out.append(("B",))
        elif m.group("wait"):
            if wait:
                out.extend(wait)
        elif m.group("add"):
            out.append(("W", int(m.group("aw"))))
        else:
            out.append(("W" if m.group("write") else "R", int(m.group("w") or 0)))
    return out


def _hazards(events):
    """Words written while a read of them may still be under way in another wave."""
    open_reads, bad = set(), set()
    for e in events:
        if e[0] == "B":
            open_reads.clear()
        elif e[0] == "R":
            open_reads.add(e[1])
        elif e[1] in open_reads:
            bad.add(e[1])
    return bad


def _columns():
    text = SRC.read_text()
    wait = _events(_body(text, "flow_wait2"), None)
    assert wait.count(("B",)) == 2 and ("W", 0) in wait and ("R", 0) in wait
    loop = _loop(_body(text, "flow_chain"))
    taken, passed = _events(loop, wait), _events(loop, None)
    assert taken.count(("B",)) >= 6 and len(taken) == len(passed) + len(wait)
    assert [e for e in passed if e[0] == "R"], "the early look at the hand-off flags is gone"
    return taken, passed


def test_no_word_is_rewritten_under_a_read():
    for two in itertools.product(_columns(), repeat=3):
        assert not _hazards([e for col in two for e in col])


def test_the_check_finds_a_shared_word():
    """The early look and the wait through one word: a write under a read."""
    taken, passed = _columns()
    early = [e[1] for e in passed if e[0] == "R"][-1]
    same = [(e[0], 0) if len(e) > 1 and e[1] == early else e for e in taken]
    assert _hazards(same + same) == {0}
