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


def view(buffer) -> torch.Tensor:
    """uint8 tensor over the bytes of any buffer (no copy; not to be written unless the caller owns
    the buffer)."""
    return torch.frombuffer(buffer, dtype=torch.uint8)


def new_bytes(n: int):
    """(bytes object of n > 0 bytes with undefined contents, uint8 tensor over them): to be filled
    through the tensor before anybody else sees the object."""
    b = _new(None, n)
    return b, view(b)
