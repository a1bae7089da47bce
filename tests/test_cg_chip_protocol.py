"""The all-reduce of the on-chip CG (resident_dev.hpp): its slots are used again
after kSlotGens generations, reset by their owner in between.  Every execution
of a few iterations is explored on a model in which a workgroup's stores to
different addresses are performed in any order until it waits for them; no
workgroup may take a sum of an older generation for the one it polls."""
import os
import re

import pytest

CSRC = os.path.join(os.path.dirname(__file__), "..", "mtl4_amd", "csrc")
PENDING = -1


def _source(name):
    with open(os.path.join(CSRC, name)) as f:
        return re.sub(r"//[^\n]*", "", f.read())


def _steps():
    """The kernels' waits of one iteration, in order: the same in both."""
    found = []
    for name, kernel in (("resident.hip", "k_cg_resident"), ("resident_large.hip", "k_cg_large")):
        text = _source(name)
        body = text[text.index("void %s(" % kernel):]
        body = body[:body.index("L.leave(")]
        body = body[body.rindex("for (;;)"):]
        found.append(re.findall(r"res_(exchange|allsum)\b", body))
    assert found[0] == found[1]
    return found[0]


def _program(me, groups, steps, gens, iterations):
    """Workgroup `me`'s operations: publish, poll everyone, reset the generation
    before; an exchange waits for the workgroup's own stores (it need not wait for
    any other: the modelled workgroups are no neighbours)."""
    ops, g = [], 0
    for _ in range(iterations):
        for s in steps:
            if s == "exchange":
                ops.append(("wait",))
                continue
            ops.append(("store", (g % gens, me), g))
            ops += [("poll", (g % gens, w), g) for w in range(groups)]
            ops.append(("store", ((g - 1) % gens, me), PENDING))
            g += 1
    return tuple(ops)


def _stale_read(gens, steps, groups=2, iterations=3):
    progs = [_program(w, groups, steps, gens, iterations) for w in range(groups)]
    slots = [(g, w) for g in range(gens) for w in range(groups)]
    start = (tuple([0] * groups), tuple([()] * groups), tuple([PENDING] * len(slots)))
    todo, seen = [start], {start}
    while todo:
        at, flight, mem = todo.pop()
        after = []
        for w in range(groups):
            # a store in flight is performed (stores to one address stay in order)
            for k, (addr, v) in enumerate(flight[w]):
                if any(a == addr for a, _ in flight[w][:k]):
                    continue
                m = list(mem)
                m[slots.index(addr)] = v
                f = list(flight)
                f[w] = flight[w][:k] + flight[w][k + 1:]
                after.append((at, tuple(f), tuple(m)))
            if at[w] == len(progs[w]):
                continue
            op = progs[w][at[w]]
            f = flight
            if op[0] == "wait":
                if flight[w]:
                    continue
            elif op[0] == "store":
                f = list(flight)
                f[w] = flight[w] + ((op[1], op[2]),)
                f = tuple(f)
            else:
                v = mem[slots.index(op[1])]
                if v == PENDING:
                    continue
                if v != op[2]:
                    return True
            a = list(at)
            a[w] += 1
            after.append((tuple(a), f, mem))
        for s in after:
            if s not in seen:
                seen.add(s)
                todo.append(s)
    assert any(s[0] == tuple(len(p) for p in progs) for s in seen)   # the model runs to the end
    return False


def test_no_sum_of_an_older_generation_is_read():
    m = re.search(r"constexpr int kSlotGens = (\d+);", _source("resident_dev.hpp"))
    gens = int(m.group(1)) if m else int(re.search(r"slots \+ \(size_t\)\(gen % (\d+)\)",
                                                   _source("resident_dev.hpp")).group(1))
    steps = _steps()
    assert steps == ["exchange", "allsum", "allsum"]
    assert not _stale_read(gens, steps)


@pytest.mark.parametrize("gens,steps", [(3, ["exchange", "allsum", "allsum"]), (4, ["allsum", "allsum"])])
def test_the_model_sees_a_missing_wait(gens, steps):
    assert _stale_read(gens, steps)
