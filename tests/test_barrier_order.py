"""The grid barrier of the persistent batched step (`persist_barrier`): whatever each workgroup wrote
before it happens before whatever any workgroup reads after it. The atomics and fences are read from
the kernel's source in their order and run through the C++ memory model's rules (fences,
release sequences) as vector clocks, for every order of arrival of four workgroups; a relaxed read
counts only once an acquire fence follows it. On the CPU."""
import itertools
import os
import re

import pytest

REPO = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
SOURCE = os.path.join(REPO, "morphogenesis_amd", "csrc", "mg_kernels.hip")
OP = re.compile(
    r"__builtin_amdgcn_fence\(__ATOMIC_(?P<fence>\w+), \"(?P<fscope>\w+)\"\)"
    r"|__hip_atomic_(?P<op>fetch_add|store|load)\(&ctl->(?P<at>count|sense)\b[^;]*?__ATOMIC_(?P<order>\w+), __HIP_MEMORY_SCOPE_(?P<scope>\w+)\)")


def barrier():
    """(common ops, the last arriver's, the waiters', common ops after) of thread 0."""
    text = open(SOURCE).read()
    start = text.index("void persist_barrier(")
    body = text[start:text.index("\n}\n", start)]
    body = re.sub(r"/\*.*?\*/", "", body, flags=re.S)
    head, rest = body.split("if (arrived == gridDim.x) {")
    last, rest = rest.split("} else {")
    end = re.search(r"\n        }\n", rest).start()
    parts = [[m.groupdict() for m in OP.finditer(t)] for t in (head, last, rest[:end], rest[end:])]
    for m in itertools.chain(*parts):
        assert (m["fscope"] or m["scope"].lower()) == "agent", "every workgroup of the GPU takes part"
    return parts


def join(a, b):
    return [max(x, y) for x, y in zip(a, b)]


class Group:
    """One workgroup's view: `now` what happens before its next operation, `rel` that at its last
    release fence, `acq` what its relaxed reads will bring at the next acquire fence."""

    def __init__(self, k, n):
        self.now = [0] * n
        self.now[k] = 1  # its writes before the barrier
        self.rel, self.acq = [0] * n, [0] * n

    def run(self, ops, memory):
        for m in ops:
            if m["fence"]:
                if m["fence"] in ("RELEASE", "ACQ_REL"):
                    self.rel = list(self.now)
                if m["fence"] in ("ACQUIRE", "ACQ_REL"):
                    self.now = join(self.now, self.acq)
                continue
            was = memory[m["at"]]
            if m["op"] != "store":
                self.acq = join(self.acq, was)
                if m["order"] in ("ACQUIRE", "ACQ_REL"):
                    self.now = join(self.now, was)
            if m["op"] != "load":
                out = self.now if m["order"] in ("RELEASE", "ACQ_REL") else self.rel
                # a read-modify-write continues the release sequence it reads from
                memory[m["at"]] = join(was, out) if m["op"] == "fetch_add" else list(out)


@pytest.mark.parametrize("n", [2, 3, 4])
def test_every_write_happens_before_every_read(n):
    head, last, wait, tail = barrier()
    assert [m["op"] for m in head if m["op"]] == ["fetch_add"] and any(m["at"] == "sense" for m in last)
    for order in itertools.permutations(range(n)):
        memory = {"count": [0] * n, "sense": [0] * n}
        groups = [Group(k, n) for k in range(n)]
        for k in order:
            groups[k].run(head, memory)
        groups[order[-1]].run(last + tail, memory)
        for k in order[:-1]:
            groups[k].run(wait + tail, memory)
        for k in range(n):
            assert groups[k].now == [1] * n, f"arrivals {order}: workgroup {k} sees {groups[k].now}"
