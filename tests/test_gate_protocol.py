"""The gate words of a layer-tail launch under any start order of its workgroups (a model of gate_arrive, gate_wait and
the go value in csrc/layer_tail.h; the word that the go value is read from is taken from the source)."""
import random
import re
from pathlib import Path

import pytest

SRC = (Path(__file__).resolve().parent.parent / "estudiocanciones_amd" / "csrc" / "layer_tail.h").read_text()
NB, GATE_FLAGS = 64, 1024
PER = NB // 8


def start_word_of_the_source():
    """x -> word index, from the expression of GATE_START; both kernels read their go value there."""
    expr = re.search(r"constexpr int GATE_START\(int x\) \{ return (.*?); \}", SRC).group(1)
    reads = re.findall(r"if \(ld0\) go = ld_sc1\((.*)\);", SRC)
    assert len(reads) == 2 and all(re.fullmatch(r"a0?\.sync \+ GATE_START\(blockIdx\.x & 7\)", r) for r in reads)
    return lambda x: eval(expr, {"GATE_FLAGS": GATE_FLAGS, "x": x})


def workgroup(b, mem, start, gates, head, epochs):
    """One workgroup's loader, one memory access per step; a generator that yields between them."""
    grp = b % 8
    go = mem[start(grp)]
    yield
    for gate in range(1 if head else gates):
        mem[64 * (1 + grp)] = mem.get(64 * (1 + grp), 0) + 1
        if mem[64 * (1 + grp)] == (go + 1) * PER:
            yield
            for x in range(8):
                mem[GATE_FLAGS + 32 * (8 * x + grp)] = go + 1
        yield
        if not head:  # a head launch arrives and does not wait
            while any(mem[GATE_FLAGS + 32 * (8 * grp + g)] < go + 1 for g in range(8)):
                yield "wait"
        go += 1
    epochs[b] = go


def run(start, late, gates=3, launches=("head", "tail", "tail"), seed=0):
    """Launches in turn on one gate region; workgroup `late` starts only when nothing else can move.  The epochs of each
    launch, or None where it does not end."""
    rng = random.Random(seed)
    mem = {GATE_FLAGS + 32 * i: 0 for i in range(64)}
    out = []
    for kind in launches:
        epochs = {}
        wgs = {b: workgroup(b, mem, start, gates, kind == "head", epochs) for b in range(NB)}
        held, idle = {late}, 0
        while wgs:
            ready = [b for b in wgs if b not in held]
            if held and (not ready or idle > 20 * NB):
                held, idle = set(), 0
                continue
            if idle > 200 * NB:  # only waits, however often each has looked
                return out + [None]
            b = rng.choice(ready)
            try:
                idle = idle + 1 if next(wgs[b]) == "wait" else 0
            except StopIteration:
                del wgs[b]
                idle = 0
        out.append(epochs)
    return out


def sound(result):
    return all(e is not None and len(set(e.values())) == 1 and len(e) == NB for e in result)


@pytest.mark.parametrize("late", [0, 3, 8, 21, 63])
def test_a_late_workgroup_holds_the_same_go_value(late):
    start = start_word_of_the_source()
    for seed in range(5):
        assert sound(run(start, late, seed=seed))


def test_the_model_sees_a_go_value_from_another_group():
    """Read from group 0's flag, a late workgroup of another group starts one gate ahead."""
    assert not sound(run(lambda x: GATE_FLAGS + 32 * 8 * x, 3))
    assert not sound(run(lambda x: GATE_FLAGS + 32 * 8 * x, 3, launches=("tail", "tail")))
    assert sound(run(lambda x: GATE_FLAGS + 32 * 8 * x, 8))  # a workgroup of group 0 itself
