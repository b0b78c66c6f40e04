"""Copies between ordinary and pinned memory by several threads (cg_host_fill), on the CPU: the mark is an ordinary
word that the test sets."""
import concurrent.futures
import ctypes
import os
import struct
import subprocess
import sys
import threading
import time

import pytest
import torch

from cachegen_amd import _lib, hostmem

PART = struct.Struct("<3q2i")


def team(threads):
    """CgHostTeam of so many threads; 0: none."""
    return struct.pack("<2Q2i", *hostmem._openmp(), threads, 0) if threads else None


def fill(parts, mark, threads):
    raw = b"".join(PART.pack(d.data_ptr(), s.data_ptr(), d.numel(), v, 0) for d, s, v in parts)
    _lib.check(_lib.lib().cg_host_fill(raw, len(parts), mark.data_ptr(), team(threads), None))


def test_torchs_threads_are_found():
    parallel, number, threads, _ = struct.unpack("<2Q2i", hostmem.team())
    assert parallel and number and threads == torch.get_num_threads()


def data(n, seed):
    return torch.randint(0, 256, (n,), generator=torch.Generator().manual_seed(seed), dtype=torch.uint8)


# nothing, a byte, either side of a block, blocks dealt to more threads than there are
@pytest.mark.parametrize("threads", [0, 1, 3, 64])
@pytest.mark.parametrize("sizes", [(0, 1), ((64 << 10) - 1, 64 << 10, (64 << 10) + 1), (5, (3 << 20) + 17, 0, 300001)])
def test_parts_are_copied(threads, sizes):
    src = [data(n + 3, n)[3:] for n in sizes]
    room = torch.full((sum(sizes) + 7 * len(sizes) + 1,), 9, dtype=torch.uint8)
    dst, at = [], 1
    for n in sizes:
        dst.append(room[at:at + n])
        at += n + 7
    mark = torch.zeros(1, dtype=torch.int32)
    fill([(d, s, 0) for d, s in zip(dst, src)], mark, threads)
    assert all(torch.equal(d, s) for d, s in zip(dst, src))
    assert int((room == 9).sum()) >= 7 * len(sizes) + 1                     # nothing between the parts was written
    keep = torch.ones_like(room, dtype=torch.bool)
    at = 1
    for n in sizes:
        keep[at:at + n] = False
        at += n + 7
    assert (room[keep] == 9).all()


# either side of the size from which stores go past the caches, with parts that begin and end at any place of a line
@pytest.mark.parametrize("threads", [0, 3])
@pytest.mark.parametrize("more", [-1, 0])
def test_large_jobs_are_copied(threads, more):
    small = list(range(1, 140))
    test_parts_are_copied(threads, (*small, (8 << 20) + more - sum(small)))


@pytest.mark.parametrize("threads", [1, 6])
def test_a_part_is_read_only_when_it_has_arrived(threads):
    n = 400000
    want = [data(n, i) for i in range(4)]
    src = [torch.zeros(n, dtype=torch.uint8) for _ in want]
    dst = [torch.zeros(n, dtype=torch.uint8) for _ in want]
    mark = torch.zeros(1, dtype=torch.int32)
    word = ctypes.c_int32.from_address(mark.data_ptr())

    def arrive():
        for i, w in enumerate(want):
            time.sleep(0.002)
            src[i].copy_(w)
            word.value = i + 1
    t = threading.Thread(target=arrive)
    t.start()
    fill([(d, s, i + 1) for i, (d, s) in enumerate(zip(dst, src))], mark, threads)
    t.join()
    assert all(torch.equal(d, w) for d, w in zip(dst, want))


def test_callers_side_by_side():
    """Several jobs at once, some of them waiting for their marks."""
    wrong = []

    def caller(i):
        mark = torch.zeros(1, dtype=torch.int32)
        word = ctypes.c_int32.from_address(mark.data_ptr())
        for k in range(10):
            s, d = data(200000 + 977 * i, 31 * i + k), torch.zeros(200000 + 977 * i, dtype=torch.uint8)
            late = threading.Timer(0.001, lambda v=k + 1: setattr(word, "value", v))
            late.start()
            try:
                fill([(d[:100000], s[:100000], k), (d[100000:], s[100000:], k + 1)], mark, 4)
            except RuntimeError as e:
                wrong.append((i, k, e))
            late.join()
            if not torch.equal(d, s):
                wrong.append((i, k))
    callers = [threading.Thread(target=caller, args=(i,)) for i in range(6)]
    for c in callers:
        c.start()
    for c in callers:
        c.join()
    assert not wrong


def _refuse_bad_parts():
    mark = torch.zeros(1, dtype=torch.int32)
    with pytest.raises(RuntimeError, match="bad part"):
        _lib.check(_lib.lib().cg_host_fill(PART.pack(0, 0, 5, 0, 0), 1, mark.data_ptr(), None, None))
    with pytest.raises(RuntimeError, match="nothing to copy"):
        _lib.check(_lib.lib().cg_host_fill(PART.pack(0, 0, 0, 0, 0), 0, mark.data_ptr(), None, None))
    with pytest.raises(RuntimeError, match="too small"):
        _lib.check(_lib.lib().cg_host_stage(PART.pack(0, 0, 0, 0, 0), 0, (ctypes.c_void_p * 1)(64), 1, 64, 64, 1000, mark.data_ptr(), 0, None, ctypes.byref(ctypes.c_int()), None))


def test_bad_parts_are_refused():
    with concurrent.futures.ThreadPoolExecutor(1) as other:                 # the last error's text belongs to a thread
        other.submit(_refuse_bad_parts).result()


class ShortTeam:
    """A runtime that is asked for a team and gives `given` threads, the caller among them."""

    def __init__(self, given):
        self.given, self.numbers = given, {}
        self.member = ctypes.CFUNCTYPE(None, ctypes.c_void_p)
        self._parallel = ctypes.CFUNCTYPE(None, ctypes.c_void_p, ctypes.c_void_p, ctypes.c_uint, ctypes.c_uint)(self.parallel)
        self._number = ctypes.CFUNCTYPE(ctypes.c_int)(lambda: self.numbers[threading.get_ident()])

    def parallel(self, fn, data, threads, flags):
        def run(i):
            self.numbers[threading.get_ident()] = i
            self.member(fn)(data)
        others = [threading.Thread(target=run, args=(i,)) for i in range(1, min(threads, self.given))]
        for t in others:
            t.start()
        run(0)
        for t in others:
            t.join()

    def packed(self, asked):
        return struct.pack("<2Q2i", *(ctypes.cast(f, ctypes.c_void_p).value for f in (self._parallel, self._number)), asked, 0)


def stage(lib, size, step, slots, asked, given, order=1):
    """Whether all of `size` bytes arrive, staged by `given` threads where `asked` were dealt blocks."""
    g = torch.Generator().manual_seed(size)
    want = torch.randint(0, 256, (size,), generator=g, dtype=torch.uint8)
    cuts = sorted({0, size, *(int(x) for x in torch.randint(0, size, (5,), generator=g))})
    area = torch.zeros(size, dtype=torch.uint8)
    pinned = [torch.empty(step, dtype=torch.uint8) for _ in range(slots)]
    raw = b"".join([PART.pack(a, want[a:].data_ptr(), b - a, 0, 0) for a, b in zip(cuts, cuts[1:])][::order])
    team, moves = ShortTeam(given), ctypes.c_int(0)
    rc = lib.cg_test_host_stage(raw, len(cuts) - 1, (ctypes.c_void_p * slots)(*(t.data_ptr() for t in pinned)), slots, step,
                                area.data_ptr(), size, team.packed(asked) if given else None, ctypes.byref(moves))
    return rc == 0 and torch.equal(area, want) and moves.value == -(-size // step) + 1


def stage_all():
    """Pinned slots in turn, two and four of them, sizes in and above the ring; the caller alone, fewer threads than were asked
    for, as many; parts that do not ascend."""
    lib = _lib.lib()
    for asked, given in ((8, 0), (1, 1), (8, 1), (8, 2), (8, 4), (16, 3), (8, 8)):
        for slots in (2, 4):
            for step, size in ((64, 1000), (256 << 10, (256 << 10) * slots), (256 << 10, (3 << 20) + 77), (1 << 20, (9 << 20) + 1)):
                print(asked, given, slots, step, size, flush=True)
                assert stage(lib, size, step, slots, asked, given)
    assert stage(lib, (3 << 20) + 77, 256 << 10, 4, 8, 4, order=-1)


def test_staged_uploads_end_with_any_team():
    """In a process of its own, which a job that does not end would not leave."""
    done = subprocess.run([sys.executable, "-c", "import test_threaded_copy as t; t.stage_all()"], timeout=100, capture_output=True, text=True,
                          env={**os.environ, "PYTHONPATH": os.pathsep.join([os.path.dirname(__file__), os.path.dirname(os.path.dirname(__file__))])})
    assert done.returncode == 0, done.stdout[-500:] + done.stderr[-2000:]
