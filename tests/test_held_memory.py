"""Pinned memory on its way up (hostmem.Moves.hold): the bound on all of it, and who waits for whom.  On the CPU, with events
that the test lets through."""
import collections
import random
import threading

import pytest
import torch

from cachegen_amd import hostmem

LIMIT = 1 << 20


class Event:
    def __init__(self, waits=True):
        self.through, self.waited, self.waits = threading.Event(), 0, waits

    def query(self):
        return self.through.is_set()

    def synchronize(self):
        self.waited += 1
        assert self.waits, "waited for another stream's work"
        self.through.set()


@pytest.fixture(autouse=True)
def nothing_held(monkeypatch):
    monkeypatch.setattr(hostmem, "_HELD_BYTES", LIMIT)
    monkeypatch.setattr(hostmem, "_held", collections.deque())
    monkeypatch.setattr(hostmem, "_held_bytes", 0, raising=False)
    monkeypatch.setattr(hostmem, "_events", {})


def hold(size, event, stream=1):
    moves = object.__new__(hostmem.Moves)
    moves.device, moves.stream = torch.device("cuda", 0), stream
    moves._going_up, moves._count = [torch.empty(size, dtype=torch.uint8)], 1
    moves.hold(event)
    return event


def held():
    return sum(t.numel() for h in hostmem._held for t in h[-1])


def test_a_small_oldest_entry_does_not_let_larger_ones_through():
    first = hold(16, Event())
    events = [hold(400 << 10, Event()) for _ in range(6)]
    assert held() <= LIMIT
    assert first.through.is_set() and events[0].through.is_set() and not events[-1].through.is_set()


def test_the_bound_holds_for_any_sizes():
    rnd = random.Random(1)
    for k in range(300):
        hold(rnd.choice([0, 1, 1000, 300 << 10, LIMIT - 1, LIMIT, LIMIT + 1, 3 * LIMIT]), Event(), stream=rnd.randrange(3))
        assert held() <= LIMIT
        for h in list(hostmem._held):
            if rnd.random() < 0.2:
                h[0].through.set()


def test_nobody_waits_for_another_streams_work():
    """A stream that stands still: others go on, and what of theirs is through is given back."""
    hold(LIMIT - 10, Event(waits=False), stream=1)
    for k in range(4):
        mine = hold(LIMIT // 2, Event(), stream=2)
        assert mine.waited == 1 and held() <= LIMIT
    later = hold(5, Event(), stream=2)
    later.through.set()
    hostmem._let_all_go()
    assert held() == LIMIT - 10 and len(hostmem._events[0]) <= 16


def test_others_are_not_held_up_by_a_wait():
    """The wait is not made under the lock that every call takes."""
    waiting, go = threading.Event(), threading.Event()

    class Slow(Event):
        def synchronize(self):
            waiting.set()
            assert go.wait(20)
            self.through.set()
    t = threading.Thread(target=lambda: hold(2 * LIMIT, Slow(), stream=1))
    t.start()
    assert waiting.wait(20)
    assert hostmem._held_lock.acquire(timeout=5)
    hostmem._held_lock.release()
    go.set()
    t.join()
    assert held() == 0


def test_memory_that_has_been_read_serves_the_next_allocation(monkeypatch):
    """Not only the next upload: torch's pool would get new memory from the system for what comes down meanwhile."""
    given = []
    monkeypatch.setattr(torch, "empty", lambda *size, pin_memory=False, **kw: given.append(held()) or torch.zeros(*size, **kw))
    first, second = hold(1000, Event()), hold(2000, Event())
    given.clear()
    first.through.set()
    assert hostmem.pinned(64).shape == (64,) and given.pop() == 2000
    second.through.set()
    device = torch.device("cpu")
    hostmem.Moves(device, 0).room(torch.zeros(8))
    assert given.pop() == 0
