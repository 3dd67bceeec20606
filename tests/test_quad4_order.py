"""CPU test: the counted waits of k_quad4 hold for every order the compiler may choose.

The kernel waits by count: the copy of a record into LDS has landed when at most
so many younger memory operations are in flight. A load that no fence keeps in
place may be issued earlier than written. The test reads the kernel's source for
its operations (copies, the load of the next words, fences, waits), issues the
load of the words at the earliest place its fences allow, and checks at every
wait that the record read next is among the operations retired in issue order.
"""
import os
import re

SRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "conquest-release_amd", "csrc",
                   "cq_tile.hip")
TOKENS = re.compile(r'(?P<copy>\bcopy\()|(?P<words>=\s*words\[8 \*)|(?P<fence>asm volatile\("" ::: "memory"\))'
                    r'|(?P<wait>s_waitcnt\((?P<count>\(?AHEAD[^|]*)\|)')


def _tokens(text):
    return [(m.lastgroup if m.lastgroup != "count" else "wait", m.group("count")) for m in TOKENS.finditer(text)]


def _issue_order(events):
    """The events with each load of the words moved up to the fence before it."""
    out = []
    for ev in events:
        at = len(out)
        if ev[0] == "words":
            while at > 0 and out[at - 1][0] not in ("fence", "wait"):
                at -= 1
        out.insert(at, ev)
    return out


def test_copies_have_landed_at_every_wait():
    text = open(SRC).read()
    body = text[text.index("k_quad4(const ARG arg)"):]
    body = body[:body.index("// FP64 accumulator D[g+4e][r]")]
    ahead = int(re.search(r"AHEAD = (\d+);", body).group(1))
    start = body.index("i < AHEAD; ++i) copy(w, i, i);")
    loop = body.index("for (int32_t rec = 0;")
    inner = body.index("for (int i = 0; i < 8; ++i)", loop)
    end = body.index("w = wn;", inner)
    assert [k for k, _ in _tokens(body[start:loop])] == ["copy"]
    head = _tokens(body[loop:inner])
    each = _tokens(body[inner:end])
    assert [k for k, _ in head if k != "fence"] == ["words"]
    assert [k for k, _ in each if k != "fence"] == ["copy", "wait", "wait"]
    waits = [eval(c, {"AHEAD": ahead}) for k, c in each if k == "wait"]  # first AHEAD records, the others

    events = [("copy", r) for r in range(ahead)]
    for rec in range(0, 32, 8):
        events += [(k, rec) for k, _ in head]
        for i in range(8):
            done = False
            for k, _ in each:
                if k == "wait":
                    if not done:
                        events.append(("wait", (rec + i, waits[0] if i < ahead else waits[1])))
                    done = True
                else:
                    events.append((k, rec + i + ahead))
    flying = []
    for k, v in _issue_order(events):
        if k in ("copy", "words"):
            flying.append((k, v))
        elif k == "wait":
            record, count = v
            flying = flying[max(0, len(flying) - count):]
            assert ("copy", record) not in flying, f"record {record} is read with its copy in flight"
