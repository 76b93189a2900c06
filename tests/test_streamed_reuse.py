"""When k_bicg_streamed (csrc/isph_streamed.hip) may overwrite the vectors
that its blocks read from each other.

The test takes the stores, loads and exchanges of an iteration from the kernel
source, in order, with the arrays that v and t go to, and walks every order in
which two blocks can pass them: a block passes an exchange once both have
published their part of it.  What an exchange's `between` reads counts as read
after the wait, as other waves than the waiting one run it.  Every load must
find the value of its own iteration.
"""
import os
import re

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
ITERATIONS = 5


def kernel_events():
    """Events of an iteration: ("store" | "load", vector), ("publish",),
    ("wait",); and the array of each vector by iteration parity."""
    path = os.path.join(ROOT, "beach_slope_confined_amd", "csrc", "isph_streamed.hip")
    text = re.sub(r"//[^\n]*", "", open(path).read())
    kernel = text[text.index("k_bicg_streamed(KrylovArgs"):text.index("namespace host")]
    arrays = {}
    for name, odd, even, fixed in re.findall(
            r"TX\* (?:const )?(\w+) = (?:it & 1 \? (a\.\w+) : (a\.\w+)|(a\.\w+));", kernel):
        arrays[name] = (fixed, fixed) if fixed else (even, odd)
    body = kernel[kernel.index("for (int it = 0;"):]
    between = {"idle": []}
    m = re.search(r"auto (\w+) = \[&\] \{.*?\n        \};", body, flags=re.S)
    between[m.group(1)] = [("load", v) for v in re.findall(r"gs_load\((\w+) \+", m.group(0))]
    body = body.replace(m.group(0), "")
    events = []
    for m in re.finditer(r"gs_(store|load)\((\w+) \+|st_exchange\(([^;]*?)\)\)", body):
        if m.group(1):
            events.append((m.group(1), m.group(2)))
        else:
            events += [("publish",), ("wait",)] + between[m.group(3).split(",")[-1].strip()]
    return events, arrays


def test_no_block_overwrites_what_another_still_reads():
    events, arrays = kernel_events()
    kinds = [e[0] for e in events]
    assert kinds.count("wait") == 3 and kinds.count("store") == 2 and kinds.count("load") == 3
    program = []  # (kind, array, tag) over the iterations; a tag is (vector, iteration)
    for it in range(ITERATIONS):
        for e in events:
            if len(e) == 2:
                program.append((e[0], arrays[e[1]][it & 1], (e[1], it)))
            else:
                program.append((e[0], None, None))
    published = [sum(p[0] == "publish" for p in program[:k]) for k in range(len(program) + 1)]
    memory, now = [], {}  # a block's arrays after its first k events
    for p in program + [("end", None, None)]:
        memory.append(dict(now))
        if p[0] == "store":
            now[p[1]] = p[2]
    seen, todo = {(0, 0)}, [(0, 0)]
    while todo:
        state = todo.pop()
        for b in (0, 1):
            at, other = state[b], state[1 - b]
            if at == len(program):
                continue
            kind, array, tag = program[at]
            if kind == "wait" and published[other] < published[at]:
                continue
            if kind == "load":
                found = memory[other].get(array)
                assert found == tag, f"{tag} read as {found}"
            nxt = (at + 1, other) if b == 0 else (other, at + 1)
            if nxt not in seen:
                seen.add(nxt)
                todo.append(nxt)
    assert (len(program), len(program)) in seen
