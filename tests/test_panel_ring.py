"""CPU: the ring of panel buffers of the weight walk (csrc/panel_ring.hpp, the very rule the kernel waits by).  Every order in
which the fetching and the multiplying waves can run is walked through: no panel is read or overwritten while one is still on its
way into its buffer, and no wave waits for ever, whichever panels no wave of a set has a block in."""
import functools
import itertools
import random

import pytest

import lds_bank_model

STEPS = 9
lib = lds_bank_model.index_lib()
READY, DONE, FETCHERS = lib.bsa_panel_ready(), lib.bsa_panel_done(), lib.bsa_panel_fetchers()
ROW_TILES = (2, 3, 4, 5)                         # what a launch chooses from


def watched(s, stages, walkers):
    """Flags that the fetch of panel s waits for, and the value they have to reach."""
    return {lib.bsa_panel_refill_flag(lane, walkers, s, stages) for lane in range(64)}, lib.bsa_panel_refill_from(s, stages)


def read_by_all(s, stages, walkers):
    """The rule without the second half: that the panel before has arrived."""
    return {DONE + w for w in range(walkers)}, s - stages + 1


def faults(stages, fetchers, needs, rule, steps=STEPS):
    """What can happen, of "overwritten" (two fetches on their way into one buffer), "read early" (or a panel that is not the
    wanted one) and "stuck".  ``needs``: the panels each multiplying wave has blocks in, ascending.  A fetching wave waits by
    ``rule``, requests, waits for what it requested, stores its flag; a multiplying wave stores how far it is done, waits for the
    next panel it needs, reads it.  A fetch writes at any time between its request and its arrival."""
    gates = [rule(s, stages, len(needs)) for s in range(steps)]
    flags = [0] * (DONE + len(needs))
    start = (tuple(flags), (-1,) * stages, tuple((f, 0) for f in range(fetchers)), tuple((0, 0) for _ in needs))
    seen, todo, found = {start}, [start], set()
    while todo:
        flags, held, fetch, walk = todo.pop()
        moves = []

        def move(flag=None, buffer=None, f=None, w=None):
            put = lambda values, change: values if change is None else values[:change[0]] + (change[1],) + values[change[0] + 1:]
            moves.append((put(flags, flag), put(held, buffer), put(fetch, f), put(walk, w)))

        flying = [s % stages for s, phase in fetch if phase == 1]
        if len(set(flying)) < len(flying):
            found.add("overwritten")
        if any(phase == 2 and (needs[w][i] % stages in flying or held[needs[w][i] % stages] != needs[w][i])
               for w, (i, phase) in enumerate(walk)):
            found.add("read early")
            continue
        for f, (s, phase) in enumerate(fetch):
            if s >= steps:
                continue
            if phase == 0 and all(flags[x] >= gates[s][1] for x in gates[s][0]):
                move(f=(f, (s, 1)))
            elif phase == 1:
                move(f=(f, (s, 2)), buffer=(s % stages, s))
            elif phase == 2:
                move(f=(f, (s + fetchers, 0)), flag=(READY + s % stages, s + 1))
        for w, (i, phase) in enumerate(walk):
            if phase == 0:                                              # done with all before its next panel, or with all there are
                move(w=(w, (i, 1)), flag=(DONE + w, needs[w][i] if i < len(needs[w]) else steps))
            elif i < len(needs[w]) and phase == 1 and flags[READY + needs[w][i] % stages] >= needs[w][i] + 1:
                move(w=(w, (i, 2)))
            elif i < len(needs[w]) and phase == 2:
                move(w=(w, (i + 1, 0)))
        if not moves and not (all(s >= steps for s, _ in fetch) and all(i == len(n) and p == 1 for n, (i, p) in zip(needs, walk))):
            found.add("stuck")
        for state in moves:
            if state not in seen:
                seen.add(state)
                todo.append(state)
    return found


def some_panels(rng):
    return tuple(sorted(rng.sample(range(STEPS), rng.randint(0, STEPS))))


def sizes():
    return sorted({(lib.bsa_panel_stages(rt), FETCHERS) for rt in ROW_TILES})


def test_the_ring_is_as_large_as_what_the_test_reckons_with():
    assert sizes() == [(3, 3), (4, 3)] and READY + 4 <= DONE


@pytest.mark.parametrize("stages,fetchers", sizes())
def test_one_wave_with_any_panels(stages, fetchers):
    for n in range(STEPS + 1):
        for needs in itertools.combinations(range(STEPS), n):
            assert faults(stages, fetchers, [needs], watched) == set(), needs


@pytest.mark.parametrize("stages,fetchers", sizes())
def test_two_waves(stages, fetchers):
    rng = random.Random(stages)
    fixed = [[(1, 4, 5, 8), ()], [(0, 8), (3, 4)], [(), ()], [tuple(range(STEPS)), (8,)]]
    for needs in fixed + [[some_panels(rng), some_panels(rng)] for _ in range(12)]:
        assert faults(stages, fetchers, needs, watched) == set(), needs


def test_what_a_wave_did_not_wait_for_need_not_be_there():
    """The walk above finds both faults of the rule without its second half, and only where another wave refills a buffer."""
    skips, all_panels = (1, 4, 5, 8), tuple(range(STEPS))
    assert faults(4, 3, [skips], read_by_all) == {"overwritten", "read early", "stuck"}
    assert faults(4, 3, [skips, ()], read_by_all) == {"overwritten", "read early", "stuck"}
    assert faults(4, 3, [all_panels], read_by_all) == set()
    assert faults(3, 3, [skips], read_by_all) == set()
    assert faults(4, 4, [skips], read_by_all) == set()
