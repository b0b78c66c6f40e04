"""Host memory of the containers: bytes objects that are filled in place, and byte buffers seen as
tensors.

A blob that goes into or comes out of a store is a Python bytes object of several megabytes.  It
is copied from and to pinned memory by torch's own copy, which runs on its thread pool and without
the interpreter lock: 6 MB in 16 us warm and 45 us out of memory the GPU has just written, where
one thread (numpy, bytes()) takes 80 and 200."""
import ctypes
import warnings

import torch

_new = ctypes.pythonapi.PyBytes_FromStringAndSize
_new.restype = ctypes.py_object
_new.argtypes = [ctypes.c_void_p, ctypes.c_ssize_t]

# torch warns once per process that it cannot keep a tensor over a read-only buffer from being
# written: the tensors below are written only where the buffer was made for it (new_bytes)
with warnings.catch_warnings():
    warnings.simplefilter("ignore")
    torch.frombuffer(b"\0", dtype=torch.uint8)


_libc = ctypes.CDLL(None)
_libc.madvise.argtypes = [ctypes.c_void_p, ctypes.c_size_t, ctypes.c_int]
_libc.mincore.argtypes = [ctypes.c_void_p, ctypes.c_size_t, ctypes.c_void_p]
_MADV_HUGEPAGE = 14
_PAGE = 4096
_HUGE_PAGE = 2 << 20


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
    copy wait for the zeroing of the same page).  A 15 MB pickle blob made and dropped: 0.95 ms
    without, 0.55 with; a blob that gets memory used before is not written twice (54 MB in nine blobs
    of a store: 0.5 ms more if it were)."""
    b = _new(None, n)
    t = view(b)
    if n >= 2 * _HUGE_PAGE:
        at = t.data_ptr()
        first, last = -(-at // _HUGE_PAGE) * _HUGE_PAGE, (at + n) // _HUGE_PAGE * _HUGE_PAGE
        present, fresh = ctypes.c_ubyte(), 0
        for page in range(first, last, _HUGE_PAGE):
            fresh += _libc.mincore(page + _HUGE_PAGE - _PAGE, _PAGE, ctypes.byref(present)) == 0 and not present.value & 1
        if 2 * fresh * _HUGE_PAGE > last - first:
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

    def stored(self):
        """Everything that stores to the words has been launched: `read` waits for that, and not for
        what is launched afterwards.  (To be left out where nothing is: the event costs a few
        microseconds.)"""
        self._stored = self._stream.record_event()

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
