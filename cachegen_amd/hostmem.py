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
_MADV_HUGEPAGE = 14
_HUGE_PAGE = 2 << 20


def view(buffer) -> torch.Tensor:
    """uint8 tensor over the bytes of any buffer (no copy; not to be written unless the caller owns
    the buffer)."""
    return torch.frombuffer(buffer, dtype=torch.uint8)


def uninitialized(n: int) -> bytes:
    """Bytes object of n bytes with undefined contents (one that is never touched takes no memory)."""
    return _new(None, n)


def new_bytes(n: int):
    """(bytes object of n > 0 bytes with undefined contents, uint8 tensor over them): to be filled
    through the tensor before anybody else sees the object.  Memory that is fresh from the system is
    asked for in huge pages: a page fault per 4 KB costs more than the copy (a 14 MB blob made
    and dropped again: 0.81 ms in small pages, 0.50 in huge ones; 6 MB: 0.37 and 0.31)."""
    b = _new(None, n)
    t = view(b)
    if n >= 2 * _HUGE_PAGE:
        at = t.data_ptr()
        first, last = -(-at // _HUGE_PAGE) * _HUGE_PAGE, (at + n) // _HUGE_PAGE * _HUGE_PAGE
        _libc.madvise(first, last - first, _MADV_HUGEPAGE)
    return b, t
