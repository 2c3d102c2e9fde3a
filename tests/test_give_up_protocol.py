"""How the wavefronts of a workgroup that exchanges lists leave their loops when the reader gives up (csrc/resident.hip and
csrc/resident_batch.hip), in every order in which they can run: nobody may be left waiting.

The model has one wavefront of each part -- a reader, the writer, one that pulls -- with the meetings of the workgroup, the LDS
counters they wait for (updated_l, done_l, without a limit) and the words go_on, as many as the kernels declare."""
import os
import re

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "bmtk_amd", "csrc")
ROUNDS = 4      # 0 .. ROUNDS, the last one the closing pull
READER, WRITER, PULLER = range(3)


def _program(part, owns, go_at_0):
    """One round of a wavefront: (operation, argument) in order; behind it the next round, or what stands at "left"."""
    look = [("meet", None), ("look", go_at_0)]
    if part == READER:
        return ([("pulled", -1), ("updated", None)] if owns else []) + [("decide", go_at_0)] + look
    if part == WRITER:
        return [("listed", 2 if owns else 1)] + look + [("pulled", 0)]
    return [("updated", None)] + look + [("done", None), ("pulled", 0)]


def _stuck(slots, owns, go_at_0):
    """A state in which somebody waits for good, or None.  A state: (per wavefront (round, place, at a meeting), done, updated,
    go_on, given up)."""
    programs = [_program(part, owns, go_at_0) for part in (READER, WRITER, PULLER)]
    LEFT, ENDED = 1000, 1001
    start = (tuple((0, 0, False) for _ in programs), 0, 0, (1,) * slots, False)
    seen, todo = {start}, [start]

    def following(state):
        waves, done, updated, go, lost = state
        out = []
        live = [w for w in waves if w[1] != ENDED]
        if live and all(w[2] for w in live):        # (a wavefront that has ended is not waited for)
            met = tuple(w if w[1] == ENDED else (w[0], ENDED if w[1] == LEFT else w[1] + 1, False) for w in waves)
            return [(met, done, updated, go, lost)]
        for i, (k, at, waits) in enumerate(waves):
            if waits or at == ENDED:
                continue

            def put(k, at, waits=False, done=done, updated=updated, go=go, lost=lost):
                out.append((waves[:i] + ((k, at, waits),) + waves[i + 1:], done, updated, go, lost))
            if at == LEFT:
                put(k, at, True)        # the last meeting
                continue
            if at == len(programs[i]):
                put(*((k + 1, 0) if k < ROUNDS else (k, LEFT)))
                continue
            op, arg = programs[i][at]
            if op == "meet":
                put(k, at, True)
            elif op == "look":
                put(k, at + 1 if (k == 0 and not arg) or go[k % slots] else LEFT)
            elif op == "decide":
                if k == 0 and not arg:
                    put(k, at + 1)
                else:
                    for gives_up in ((True,) if lost else (False, True)):
                        put(k, at + 1, go=go[:k % slots] + (int(not gives_up),) + go[k % slots + 1:], lost=gives_up)
            elif op == "updated":
                put(k, at + 1, updated=updated + (k < ROUNDS or go_at_0))
            elif op == "done":
                put(k, at + 1, done=done + 1)
            elif op == "listed":
                if k == ROUNDS or updated >= (k + 1) * arg:
                    put(k, at + 1)
            elif op == "pulled":
                if k + arg < 0 or done >= k + arg + 1:
                    put(k, at + 1)
        return out

    while todo:
        state = todo.pop()
        nexts = following(state)
        if not nexts and any(w[1] != ENDED for w in state[0]):
            return state
        for n in nexts:
            if n not in seen:
                seen.add(n)
                todo.append(n)
    return None


@pytest.mark.parametrize("owns", [False, True])
@pytest.mark.parametrize("source,kernel,go_at_0", [("resident.hip", "sim_resident_lists_kernel", False),
                                                   ("resident_batch.hip", "sim_resident_batch_kernel", True)])
def test_nobody_is_left_waiting_when_the_reader_gives_up(source, kernel, go_at_0, owns):
    with open(os.path.join(CSRC, source)) as f:
        body = f.read().split("void %s(" % kernel)[1]
    words = re.search(r"__shared__ int go_on(?:\[(\d+)\])?;", body)
    assert _stuck(int(words.group(1) or 1), owns, go_at_0) is None


def test_the_model_sees_a_word_that_is_read_late():
    """With one word for all rounds a wavefront may read the next round's in place of its own and leave without adding to done_l;
    the others wait for that.  (A reader that owns neurons waits for the pulling wavefronts first: only the writer can be late.)"""
    assert _stuck(1, False, False) is not None and _stuck(1, False, True) is not None


@pytest.mark.parametrize("source,kernel,limit", [("resident.hip", "sim_resident_lists_kernel", "kMaxSpin"),
                                                 ("resident_batch.hip", "sim_resident_batch_kernel", "kRbMaxSpin")])
def test_the_callers_limit_holds_for_every_wait(source, kernel, limit):
    """res_spin_limit, where one is given, takes the built-in limit's place in all waits for other workgroups."""
    with open(os.path.join(CSRC, source)) as f:
        body = f.read().split("void %s(" % kernel)[1].split("\n}\n")[0]
    used = [line for line in body.splitlines() if limit in line]
    assert len(used) == 1 and "s.res_spin_limit ? s.res_spin_limit : " + limit in used[0]
