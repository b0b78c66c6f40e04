"""Host memory of the containers: bytes objects that are filled in place, and byte buffers seen as
tensors.

A blob that goes into or comes out of a store is a Python bytes object of several megabytes.  It
is copied from and to pinned memory by several threads and without the interpreter lock: a call's copies as one
job in step with the bus (`Moves.fill`, `Moves.stage`; cg_host_fill, cg_host_stage), one or two small pieces by
torch's own copy.  By eight threads 6 MB take 16 us warm and 45 us out of memory the GPU has just written, where
one (numpy, bytes()) takes 80 and 200."""
import collections
import ctypes
import os
import re
import struct
import threading
import warnings

import torch

from . import _lib

_new = ctypes.pythonapi.PyBytes_FromStringAndSize
_new.restype = ctypes.py_object
_new.argtypes = [ctypes.c_void_p, ctypes.c_ssize_t]

# torch warns once per process that it cannot keep a tensor over a read-only buffer from being
# written: the tensors below are written only where the buffer was made for it (new_bytes)
with warnings.catch_warnings():
    warnings.simplefilter("ignore")
    torch.frombuffer(b"\0", dtype=torch.uint8)


_TEAM = struct.Struct("<2Q2i")           # CgHostTeam
_libc = ctypes.CDLL(None)
_libc.madvise.argtypes = [ctypes.c_void_p, ctypes.c_size_t, ctypes.c_int]
_libc.mincore.argtypes = [ctypes.c_void_p, ctypes.c_size_t, ctypes.c_void_p]
_MADV_HUGEPAGE = 14
_PAGE = 4096
_HUGE_PAGE = 2 << 20


def _openmp():
    """(GOMP_parallel, omp_get_thread_num) of the OpenMP runtime that torch has loaded, as addresses; (0, 0) where there
    is none."""
    try:
        with open("/proc/self/maps") as f:
            paths = {line.split(None, 5)[-1].strip() for line in f if re.search(r"/lib(g|i|)omp[^/]*$", line)}
        for path in sorted(paths, key=lambda p: not p.startswith(os.path.dirname(torch.__file__))):
            runtime = ctypes.CDLL(path)
            if hasattr(runtime, "GOMP_parallel") and hasattr(runtime, "omp_get_thread_num"):
                return tuple(ctypes.cast(fn, ctypes.c_void_p).value for fn in (runtime.GOMP_parallel, runtime.omp_get_thread_num))
    except OSError:
        pass
    return 0, 0


_runtime = None


def team() -> bytes:
    """CgHostTeam: torch's threads, as many as torch uses."""
    global _runtime
    if _runtime is None:
        _runtime = _openmp()
    return _TEAM.pack(*_runtime, torch.get_num_threads(), 0)


def view(buffer) -> torch.Tensor:
    """uint8 tensor over the bytes of any buffer (no copy; not to be written unless the caller owns
    the buffer)."""
    return torch.frombuffer(buffer, dtype=torch.uint8)


def new_bytes(n: int):
    """(bytes object of n > 0 bytes with undefined contents, uint8 tensor over them): to be filled
    through the tensor before anybody else sees the object.

    Memory that the allocator has just got from the system is made present here: asked for in huge
    pages (a page fault per 4 KB costs more than the copy that causes it) and written once by all
    threads at the same time (a blob is filled section by section, and the threads of one section's
    copy wait for the zeroing of the same page).  Made present and filled, 3.6, 4.5, 6 and 14 MB: 225, 244, 193 and
    261 us, left to the copies 436, 495, 646 and 1353, the kernel asked to populate the large pages alone -, 423, 377 and
    424; 2 MB, of which a large page is seldom whole, 260 and 269.  A 15 MB pickle blob made and dropped: 0.95 ms
    without, 0.55 with; a blob that gets memory used before is not written twice (54 MB in nine blobs
    of a store: 0.5 ms more if it were)."""
    b = _new(None, n)
    t = view(b)
    if n >= 3 * _HUGE_PAGE // 2:
        at = t.data_ptr()
        first, last = -(-at // _HUGE_PAGE) * _HUGE_PAGE, (at + n) // _HUGE_PAGE * _HUGE_PAGE
        present, fresh = ctypes.c_ubyte(), 0
        for page in range(first, last, _HUGE_PAGE):
            fresh += _libc.mincore(page + _HUGE_PAGE - _PAGE, _PAGE, ctypes.byref(present)) == 0 and not present.value & 1
        if 2 * fresh * _HUGE_PAGE > max(0, last - first):
            _libc.madvise(first, last - first, _MADV_HUGEPAGE)
            t.fill_(0)
    return b, t


class StoredWords:
    """Pinned words, zero at first, that kernels on the current stream store to; to be used in a
    `with` block that holds the launches.

    torch's pool of pinned memory hands a block to the next caller as soon as its tensor is gone,
    unless one of torch's own copies still uses it: of a kernel's stores it knows nothing.  So the
    words are held until the launches are through, also when the `with` block ends in an exception."""

    def __init__(self, n: int, dtype: torch.dtype):
        self.words = torch.zeros(n, dtype=dtype, pin_memory=True)
        self._stream = torch.cuda.current_stream()
        self._stored, self._through = None, False

    def __enter__(self):
        return self

    def stored(self, by=None):
        """Everything that stores to the words has been launched: `read` waits for that, and not for
        what is launched afterwards.  (To be left out where nothing is: the event costs a few
        microseconds.)  by: an `Arrival` that comes no earlier, in the place of an event."""
        self._stored = by or self._stream.record_event()

    def _wait(self):
        (self._stored or self._stream).synchronize()
        self._through = True

    def read(self):
        """The words as a list, once the launches that store to them are through."""
        self._wait()
        return self.words.tolist()

    def __exit__(self, *exc):
        if not self._through:
            self._wait()


_free = threading.local()                # words of this thread that nobody uses


class Words:
    """64 pinned bytes that kernels of one call store to, for a host that looks at their mark instead of waiting for an event
    (cg_read_words and its like); to be used in a `with` block that holds the launches and the reads.  They are
    kept for the thread's next call; where a `with` block ends in an exception and the mark is not there, until the
    process ends: something may still store to them."""
    _lost = []

    def __enter__(self):
        kept = _free.__dict__.setdefault("words", [])
        if kept:
            self._memory, self.value = kept.pop()
        else:
            self._memory, self.value = torch.zeros(8, dtype=torch.int64, pin_memory=True), 0
        self.at = self._memory.data_ptr()
        self.mark = self.at + 56
        self.value = self.value % (1 << 30) + 1
        if self.value == 1:
            self._memory[7] = 0
        return self

    def set(self, stream):
        """The mark alone, behind what the stream holds so far."""
        _lib.check(_lib.lib().cg_mark(self.mark, self.value, stream))
        self._stream = stream
        return self

    def synchronize(self):
        self.wait(self._stream)

    def wait(self, stream):
        _lib.check(_lib.lib().cg_wait_mark(self.mark, self.value, stream))

    def clear(self):
        self._memory[:2] = 0

    def numbers(self, n):
        return self._memory[:n].tolist()

    def number(self):
        return ctypes.c_float.from_address(self.at).value

    def __exit__(self, kind, *exc):
        if kind is None or ctypes.c_int32.from_address(self.mark).value >= self.value:
            _free.words.append((self._memory, self.value))
        else:
            self._lost.append(self._memory)


def read_number(tensor, index):
    """Entry `index` of a vector of int32 or int64, once what the current stream holds is through: tensor[index].item()."""
    if not tensor.is_cuda or tensor.dim() != 1 or tensor.dtype not in (torch.int32, torch.int64) or torch.cuda.is_current_stream_capturing():
        return tensor[index].item()
    n, size = tensor.shape[0], tensor.element_size()
    if not -n <= index < n:
        return tensor[index].item()                      # raises
    at = tensor.data_ptr() + index % n * tensor.stride(0) * size
    with torch.cuda.device(tensor.device), Words() as words:
        _lib.check(_lib.lib().cg_read_words(ctypes.byref(ctypes.c_void_p(at)), ctypes.byref(ctypes.c_int32(size)), 1, words.at, words.value,
                                            torch._C._cuda_getCurrentRawStream(tensor.device.index)))
        return words.numbers(1)[0]


_PART = struct.Struct("<3q2i")           # CgHostPart


# Up to so many bytes in one or two pieces are copied by torch and moved at once: 2.7 MB are in pinned memory after 11 us, and the
# host is free after 17, where the steps take it 50 and the bytes are through no sooner.
_FEW_BYTES = 4 << 20


class Arrival:
    """What was queued up to one place of a stream."""

    def __init__(self, moves, number):
        self._moves, self._number = moves, number

    def synchronize(self):
        self._moves.wait(self._number)


class Moves:
    """Bytes between pinned host memory and device memory, moved by the copy engines on one stream, and how far they
    have got: a place of the stream behind each move that is waited for, which the host looks at without waiting and, in
    native code, in step with its own copies (cg_host_fill).

    torch's pool of pinned memory knows nothing of these moves.  What comes down is waited for, at the
    latest when the `with` block ends; what goes up is handed to `hold`."""
    _watch = None

    def __init__(self, device, stream):
        self.device, self.stream = device, stream        # the stream's raw handle; the caller has made the device current
        self._word = ctypes.c_int32(0)                   # the number of the last place that the stream is through with
        self._at = ctypes.addressof(self._word)
        self._count = self._marked = self._reached = 0
        self._going_up, self._coming_down = [], []       # pinned tensors, (number, pinned tensor)

    def __enter__(self):
        return self

    def __exit__(self, *exc):
        if self._reached < self._count:
            self.wait(self._count)

    def __del__(self):
        if self._watch and _lib is not None:             # (None when the interpreter ends)
            _lib.lib().cg_watch_free(self._watch)

    def _places(self):
        if self._watch is None:
            self._watch = _lib.lib().cg_watch_new(self._at)
        return self._watch

    def queued(self):
        """What has been queued on the stream so far."""
        self._count += 1
        return Arrival(self, self._count)

    def here(self):
        """The same, and not what is queued until somebody waits."""
        arrival = self.queued()
        self._mark()
        return arrival

    def room(self, src):
        """(a tensor as it can be moved from its address on: dense, on the device; pinned uint8 tensor for its bytes, at the
        same place inside a 16-byte unit)."""
        src = src.to(self.device).contiguous()
        n, skew = src.numel() * src.element_size(), src.data_ptr() % 16
        return src, pinned(n + skew)[skew:]

    def down(self, src, place=True):
        """(pinned uint8 tensor that receives the bytes of a tensor, their arrival).  place: False for what arrives just before
        something else that is waited for (the copy engine stops for 4 us at a place)."""
        src, host = self.room(src)
        return host, self.down_to(src.data_ptr(), host, place) if host.numel() else self.queued()

    def down_to(self, src, host, place=True):
        """The same into a slice of pinned memory, from a device address."""
        arrival = self.queued()
        _lib.check(_lib.lib().cg_move_bytes(src, host.data_ptr(), host.numel(), 1, self._places() if place else None, self._count, self.stream))
        if place:
            self._marked = self._count
        self._coming_down.append((self._count, host))
        return arrival

    def fill(self, parts):
        """parts: [(uint8 tensor in ordinary memory, uint8 tensor of the same size in pinned memory, its arrival
        or None)]: copies each as it arrives."""
        if not parts:
            return
        last = max((a._number for _, _, a in parts if a is not None), default=0)
        with torch.cuda.device(self.device):
            if self._marked < last:
                self._mark()
            described = b"".join(_PART.pack(dst.data_ptr(), src.data_ptr(), dst.numel(), 0 if a is None else a._number, 0)
                                 for dst, src, a in parts)
            _lib.check(_lib.lib().cg_host_fill(described, len(parts), self._at, team(), self._places()))
        self._have(last)

    def stage(self, pieces, base, size, step, slots=0):
        """`size` bytes at the device address `base` from pieces of ordinary memory ((offset, uint8 tensor), in order): copied
        to pinned memory and moved by steps as they are there.  slots: pinned steps that are used in turn (0: as
        many as it takes)."""
        if size <= _FEW_BYTES and len(pieces) <= 2:
            host = pinned(size)
            for at, t in pieces:
                host[at:at + t.numel()].copy_(t)
            self.up(host, base)
            return
        nsteps = -(-size // step)
        if slots and slots < nsteps:
            memory = [pinned(step) for _ in range(slots)]
            places = [t.data_ptr() for t in memory]
        else:
            memory = [pinned(size)]
            places = [memory[0].data_ptr() + i * step for i in range(nsteps)]
        described = b"".join(_PART.pack(at, t.data_ptr(), t.numel(), 0, 0) for at, t in pieces)
        launched = ctypes.c_int(0)
        rc = _lib.lib().cg_host_stage(described, len(pieces), (ctypes.c_void_p * len(places))(*places), len(places), step, base, size, None, 0,
                                      team(), ctypes.byref(launched), self.stream)
        if launched.value:
            self._count += 1
            self._going_up += memory
        _lib.check(rc)

    def up(self, host, dst):
        """Pinned memory to a device address; `host` is kept until it has been read."""
        _lib.check(_lib.lib().cg_move_bytes(host.data_ptr(), dst, host.numel(), 0, None, 0, self.stream))
        self._going_up.append(host)
        return self.queued()

    def wait(self, number):
        if self._reached < number:
            with torch.cuda.device(self.device):
                if self._marked < number:
                    self._mark()
                _lib.check(_lib.lib().cg_watch_wait(self._places(), number))
            self._have(number)

    def _mark(self):
        _lib.check(_lib.lib().cg_watch_add(self._places(), self._count, self.stream))
        self._marked = self._count

    def _have(self, number):
        self._reached = max(self._reached, number)
        while self._coming_down and self._coming_down[0][0] <= number:
            del self._coming_down[0]

    def hold(self, event):
        """Keeps what is going up until `event`, recorded behind all moves; the event is `hold`'s from here on."""
        _hold(event, (self.device.index, self.stream), self._going_up)
        self._reached = self._count


_HELD_BYTES = 256 << 20                  # of pinned memory on its way up, of all threads and streams
_held = collections.deque()              # (event, (device index, stream), pinned tensors)
_held_bytes = 0
_held_lock = threading.Lock()
_events = {}                             # device index -> events that are through, to be recorded again (a new one takes 9 us)


def _hold(event, place, tensors):
    """Where that makes more than _HELD_BYTES, the oldest of the caller's own stream are waited for, one after the other, until it
    does not or they are all through: nobody waits for another stream's work, and as every caller does so, the bound holds
    when a call has returned (calls in the middle of it come on top, with what they bring)."""
    global _held_bytes
    with _held_lock:
        _held.append((event, place, tensors))
        _held_bytes += _size(tensors)
        if _held_bytes > _HELD_BYTES:
            _let_all_go()
    while True:
        with _held_lock:
            own = next((h for h in _held if h[1] == place), None)
            if _held_bytes <= _HELD_BYTES or own is None:
                return
            _held.remove(own)            # nobody else records its event again while it is waited for
        try:
            own[0].synchronize()
        except BaseException:
            with _held_lock:
                _held.appendleft(own)
            raise
        with _held_lock:
            _gone(own)


def _size(tensors):
    return sum(t.numel() * t.element_size() for t in tensors)


def _gone(held):
    global _held_bytes
    event, (device, _), tensors = held
    _held_bytes -= _size(tensors)
    if len(_events.setdefault(device, [])) < 16:
        _events[device].append(event)


def _let_go():
    """What is through and has nothing older before it, which is what a program of one stream has."""
    while _held and _held[0][0].query():
        _gone(_held.popleft())


def _let_all_go():
    """What is through of every stream: one that stands still keeps nobody else's."""
    standing = set()
    for h in list(_held):
        if h[1] in standing:
            continue
        if h[0].query():
            _held.remove(h)
            _gone(h)
        else:
            standing.add(h[1])


def pinned(n):
    """uint8 tensor of pinned memory.  What earlier uploads have read by now is given back first: torch's pool would otherwise get
    new memory from the system, which takes long and is not allowed while another thread captures a graph."""
    with _held_lock:
        _let_go()
    return torch.empty(n, dtype=torch.uint8, pin_memory=True)


def event(device):
    """An event for `hold`; gives back the pinned memory of earlier calls that has been read by now."""
    with _held_lock:
        _let_go()
        kept = _events.get(device.index)
        return kept.pop() if kept else torch.cuda.Event()
