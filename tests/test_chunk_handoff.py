"""CPU model of the chunk kernel's hand-off (kivi_decode_mfma.hip,
kivi_decode_chunk_kernel) under random interleavings of the workgroups' memory
operations, each of which completes some time after it is issued.

A workgroup stores its partial, waits until that is complete, stores its flag,
waits again, loads the segment's flags one by one, and if all hold the launch's
epoch loads the partials, folds them and clears the flags.  Whatever the order,
some workgroup folds, every fold sees this launch's partials, and all flags are
clear at the end -- also for a replay, which repeats the epoch over the same
workspace.  Without the wait after its flag a segment can stay unfolded; without
the clear a replay can fold a stale partial."""
from __future__ import annotations

import random

EPOCH = 1 << 63 | 12345


def workgroup(mem, k, n, value, folds, wait_flag=True, clear=True):
    """Yields before each step; a pending store is a closure run at its completion."""
    pending = []

    def store(key, v):
        pending.append(lambda: mem.__setitem__(key, v))

    def drain():
        while pending:
            pending.pop(0)()
            yield
    store(("part", k), value)
    yield
    yield from drain()
    store(("flag", k), EPOCH)
    yield
    if wait_flag:
        yield from drain()
    seen = True
    for i in range(n):
        # a load is served at once, ahead of stores still on their way
        seen = seen and mem.get(("flag", i)) == EPOCH
        yield
    yield from drain()
    if not seen:
        return
    got = []
    for i in range(n):
        got.append(mem.get(("part", i)))
        yield
    folds.append(got)
    if clear:
        for i in range(n):
            store(("flag", i), 0)
            yield
    yield from drain()


def launch(rng, mem, n, tag, **how):
    folds = []
    live = [workgroup(mem, k, n, (tag, k), folds, **how) for k in range(n)]
    while live:
        w = rng.choice(live) if rng.random() < 0.7 else live[0]
        if next(w, "end") == "end":
            live.remove(w)
    return folds


def test_some_workgroup_folds_and_flags_end_clear():
    rng = random.Random(3)
    for case in range(3000):
        mem, n = {}, rng.randint(2, 7)
        for replay in range(3):
            folds = launch(rng, mem, n, (case, replay))
            assert folds and all(f == [((case, replay), k) for k in range(n)] for f in folds)
            assert all(mem[("flag", k)] == 0 for k in range(n))


def test_mutants_fail():
    rng = random.Random(4)
    assert any(not launch(rng, {}, 2, 0, wait_flag=False) for _ in range(3000))
    stale = 0
    for _ in range(3000):
        mem = {}
        launch(rng, mem, 3, 0, clear=False)
        stale += any(f != [(1, k) for k in range(3)] for f in launch(rng, mem, 3, 1, clear=False))
    assert stale
