"""The reference's pickle container without its copies.

The container is a pickle of `CacheGenGPUEncoderOutput` (cachegen_basics.py:110-131 in the
reference): a few hundred bytes of structure around one torch-saved storage per tensor.  Pickling
the tensors reads every one back from the GPU by itself, and copies its bytes into a stream, into a
bytes object and into the pickle; unpickling does the same in reverse.  Here the structure goes
through the pickle module with stand-ins for the tensors, and the storages' bytes go straight
between the blob and pinned memory: the same pickle, with one copy of the bytes.

What a torch-saved storage looks like is taken from torch itself once (`_storage_template`); a
storage that looks different is left to the plain unpickler."""
import collections
import io
import pickle
import re
import struct

import numpy as np
import torch

from .. import hostmem
from . import wire
from .cachegen_basics import CacheGenGPUBytestream, CacheGenGPUEncoderOutput, _ContainerUnpickler
from .incoming import Container

_STORAGE_NAMES = {torch.uint8: "Byte", torch.int16: "Short", torch.int32: "Int", torch.float16: "Half", torch.bfloat16: "BFloat16"}
_DTYPES = {name.encode(): dtype for dtype, name in _STORAGE_NAMES.items()}
# A pickler hands bytes objects of this size and more to its file as they are, after a piece that
# ends with their opcode and length, and puts no frame around them.
_LARGE = 1 << 16
_LARGE_HEADER = b"B" + struct.pack("<I", _LARGE)


def _text(s: bytes) -> bytes:
    return b"X" + struct.pack("<I", len(s)) + s


def _storage_template():
    """(what precedes, what lies between) the parts of a torch-saved storage that vary: its type,
    key, location and size; None if torch writes something this module does not know."""
    taken = []

    class Spy(pickle.Unpickler):
        def find_class(self, module, name):
            if (module, name) == ("torch.storage", "_load_from_bytes"):
                return lambda b: taken.append(b)
            return lambda *a: None
    Spy(io.BytesIO(pickle.dumps(torch.zeros(3, dtype=torch.uint8), protocol=4))).load()
    saved = taken[0] if taken else b""
    m = re.fullmatch(rb"(?s)(.*\nByte)(Storage\nq\x01)X....(\d+)(q\x02)X\x03\0\0\0cpu(q\x03)K\x03(Ntq\x04Q\..*)X....(\d+)(q\x01a\.)\x03\0{10}", saved)
    if not m or m.group(3) != m.group(7):
        return None
    return m.group(1)[:-len("Byte")], m.group(2), m.group(4), m.group(5), m.group(6), m.group(8)


_TEMPLATE = _storage_template()
_PREFIX = None
if _TEMPLATE is not None:
    _head, _a, _b, _c, _d, _e = (re.escape(t) for t in _TEMPLATE)
    _PREFIX = re.compile(rb"(?s)" + _head + rb"(\w{3,8})" + _a + rb"X....\d{1,20}" + _b + rb"X....[a-z]{1,8}(?::\d{1,3})?" + _c
                         + rb"(?:K.|M..|J....|\x8a[\x04-\x08].{4,8}?)" + _d + rb"X....\d{1,20}" + _e + rb"(.{8})")


def _storage_prefix(dtype, location: bytes, numel: int, key: bytes) -> bytes:
    head, a, b, c, d, e = _TEMPLATE
    size = pickle.dumps(numel, protocol=2)[2:-1]            # the number's opcode, without the frame around it
    return (head + _STORAGE_NAMES[dtype].encode() + a + _text(key) + b + _text(location) + c + size + d + _text(key) + e
            + struct.pack("<q", numel))


class _Reduced:
    """Pickles as the given call."""

    def __init__(self, fn, args):
        self._as = (fn, args)

    def __reduce__(self):
        return self._as


class _Pieces:
    """File of a pickler: keeps what is written, large bytes objects as they are."""

    def __init__(self):
        self.pieces = []

    def write(self, b):
        self.pieces.append(b if type(b) is bytes else bytes(b))


class _Writer:
    """One blob: tensors are added as host memory, `finish` writes the blob.  `arrive` waits until the
    bytes of that memory are there.  The sizes are known before: where no tensor is small enough to
    stand in the pickle itself, the blob's memory is got and made present while they are on the bus
    (13.7 MB of a context of 1333 tokens: 0.63 ms of page faults beside 0.27 of transfer; to a blob
    and back 2.06-2.17 ms one after the other, 1.80-1.93 so, in turn on one machine; on another the
    two were within their runs' spread, 2.09 and 2.13)."""

    def __init__(self, location: str, arrive, fill=None):
        """fill: copies [(bytes of the blob, host memory that `arrive` waits for)], waiting for it."""
        self.location, self.arrive, self.fill = location.encode(), arrive, fill or self._fill
        self.large = {}              # id of a stand-in bytes object of _LARGE bytes -> (object, prefix, host tensor)
        self.count = 0

    def tensor(self, host, dtype, shape, there=False):
        """Stand-in for a contiguous device tensor of this type and shape whose bytes are `host`
        (uint8 tensor; `there`: without `arrive`); the bytes are read in `finish`, few of them here."""
        numel = int(np.prod(shape, dtype=np.int64))
        self.count += 1
        prefix = _storage_prefix(dtype, self.location, numel, b"%d" % self.count)
        n = len(prefix) + host.numel()
        if n >= _LARGE:
            saved = bytes(_LARGE)
            self.large[id(saved)] = (saved, prefix, host)
        else:
            if not there:
                self.arrive()
            saved = prefix + host.numpy().tobytes()
        stride, acc = [], 1
        for s in reversed(shape):
            stride.append(acc)
            acc *= s
        storage = _Reduced(torch.storage._load_from_bytes, (saved,))
        return _Reduced(torch._utils._rebuild_tensor_v2, (storage, 0, tuple(shape), tuple(reversed(stride)), False,
                                                          collections.OrderedDict()))

    def finish(self, output: CacheGenGPUEncoderOutput) -> bytes:
        f = _Pieces()
        pickle.dump(output, f, protocol=4)
        parts, seen = [], 0                              # small bytes objects and host tensors
        for p in f.pieces:
            big = self.large.get(id(p))
            if big is None:
                parts.append(p)
                continue
            _, prefix, host = big
            seen += 1
            if not parts[-1].endswith(_LARGE_HEADER):
                raise RuntimeError("pickle: a stand-in without its header")
            n = len(prefix) + host.numel()               # the stand-in's length becomes the storage's
            header = b"B" + struct.pack("<I", n) if n < 1 << 32 else b"\x8e" + struct.pack("<Q", n)
            parts[-1] = parts[-1][:-len(_LARGE_HEADER)] + header + prefix
            parts.append(host)
        if seen != len(self.large):
            raise RuntimeError("pickle: a stand-in was copied instead of passed through")
        blob, into = hostmem.new_bytes(sum(len(p) if type(p) is bytes else p.numel() for p in parts))
        raw, at, large = into.numpy(), 0, []
        for p in parts:
            if type(p) is bytes:
                raw[at:at + len(p)] = np.frombuffer(p, dtype=np.uint8)
                at += len(p)
            else:
                large.append((into[at:at + p.numel()], p))
                at += p.numel()
        self.fill(large)
        return blob

    def _fill(self, large):
        self.arrive()
        for into, host in large:
            into.copy_(host)


def can_write(enc) -> bool:
    return _TEMPLATE is not None and enc.max_bins > 0


def pack_chunks(enc):
    """One pickle blob per chunk of an `EncodedKV`, each what pickling the chunk's
    `CacheGenGPUEncoderOutput` gives."""
    L, H, D = enc.num_layers, enc.num_heads, enc.head_size
    rows, C = 2 * L, H * D
    blobs = []
    for part in wire.bring_to_host(enc, 0, enc.num_chunks):
        w = _Writer(str(enc.payload.device), part.arrive, lambda large: part.fill([(into, host, part.arrived) for into, host in large]))
        T = part.t1 - part.t0
        maxima = torch.from_numpy(np.ascontiguousarray(part.maxima).view(np.uint8).reshape(-1))
        half = maxima.numel() // 2
        chunks, at = [], 0
        per_sub = rows * C * 4
        for g, nbytes in enumerate(part.sub_bytes):
            chunks.append(CacheGenGPUBytestream(
                bytestream=w.tensor(part.payload[at:at + nbytes], torch.uint8, (nbytes,)),
                bytestream_lengths=w.tensor(part.lengths[g * per_sub:(g + 1) * per_sub], torch.int32, (rows, C)),
                ntokens=min(wire.MAX_STREAM_BYTES, T - g * wire.MAX_STREAM_BYTES)))
            at += nbytes
        out = CacheGenGPUEncoderOutput(
            chunks, w.tensor(part.tables, torch.int16, (rows, C, enc.max_bins + 1)),
            max_tensors_key=w.tensor(maxima[:half], enc.maxima.dtype, (L, T, 1), there=True),
            max_tensors_value=w.tensor(maxima[half:], enc.maxima.dtype, (L, T, 1), there=True),
            num_heads=H, head_size=D)
        blobs.append(w.finish(out))
    return blobs


# ---- reading -------------------------------------------------------------------------------
class _NotPlain(Exception):
    """The blob is not laid out the way this module reads: the plain unpickler takes it."""


_TOKEN = b"\xffstorage"
# opcodes without an argument that may stand between frames (a frame of fewer than four bytes has no
# header): memoize, tuple of one to three, reduce, append(s), build, setitem(s), stop
_BARE = frozenset(b"\x94\x85\x86\x87Rabsuet.")


def _condense(blob):
    """(the pickle with every large bytes object replaced by a token, [(start, length) of these in
    the blob])."""
    mv = memoryview(blob)
    if len(mv) < 4 or bytes(mv[:2]) != b"\x80\x04":
        raise _NotPlain("protocol")
    out, large, pos, end = [b"\x80\x04"], [], 2, len(mv)
    while pos < end:
        op = mv[pos]
        if op == 0x95:                                   # frame
            n = 9 + struct.unpack_from("<Q", mv, pos + 1)[0]
            out.append(bytes(mv[pos:pos + n]))
            pos += n
        elif op == 0x42 or op == 0x8E:                   # bytes, 32- or 64-bit length
            head = 5 if op == 0x42 else 9
            n = struct.unpack_from("<I" if op == 0x42 else "<Q", mv, pos + 1)[0]
            token = _TOKEN + struct.pack("<I", len(large))
            out.append(b"C" + bytes([len(token)]) + token)
            large.append((pos + head, n))
            pos += head + n
        elif op in _BARE:
            out.append(bytes([op]))
            pos += 1
        else:
            raise _NotPlain("opcode between frames")
    if pos != end:
        raise _NotPlain("truncated")
    return b"".join(out), large


class _Tensor:
    """A tensor of the container: its bytes in host memory."""

    def __init__(self, dtype, host, shape):
        self.dtype, self.host, self.shape = dtype, host, shape


def _storage(large, whole, b):
    """(dtype, its bytes in host memory) of a torch-saved storage: `b`, or the large one that it is a token for."""
    if type(b) is bytes and b.startswith(_TOKEN):
        start, n = large[struct.unpack_from("<I", b, len(_TOKEN))[0]]
        data = whole[start:start + n]
        head = data[:4096].numpy().tobytes()
    else:
        head, data = b[:4096], hostmem.view(b)
    m = _PREFIX.match(head)
    if not m or m.group(1) not in _DTYPES:
        raise _NotPlain("storage")
    dtype, numel = _DTYPES[m.group(1)], struct.unpack("<q", m.group(2))[0]
    data = data[m.end():]
    if data.numel() != numel * dtype.itemsize:
        raise _NotPlain("storage size")
    return dtype, data


def _tensor(storage, offset, shape, stride, *rest):
    dtype, data = storage
    acc = 1
    for s, st in zip(reversed(shape), reversed(stride)):
        if s != 1 and st != acc:
            raise _NotPlain("strides")
        acc *= s
    size = dtype.itemsize
    if offset < 0 or (offset + acc) * size > data.numel():
        raise _NotPlain("tensor outside its storage")
    return _Tensor(dtype, data[offset * size:(offset + acc) * size], tuple(shape))


class _Reader(_ContainerUnpickler):
    """Admits what `_ContainerUnpickler` admits, with tensors left where their bytes are.

    What `find_class` gives out must not lead back to the reader: it stays in the unpickler's memo, which the
    garbage collector does not look into, and the blob would stay with it for good (a context of 1333
    tokens to a blob of 13.8 MB and back 1640 us with methods of the reader here,
    each time in memory new from the system, 1289 now).  Nor is it a function of this module: a pickle may
    set the attributes of what it is given (BUILD), and those of a module's function outlive the blob."""

    def __init__(self, condensed, large, whole):
        super().__init__(io.BytesIO(condensed))
        self._given = {("torch._utils", "_rebuild_tensor_v2"): lambda *args: _tensor(*args),
                       ("torch.storage", "_load_from_bytes"): lambda *args: _storage(large, whole, *args)}

    def find_class(self, module, name):
        return self._given.get((module, name)) or super().find_class(module, name)


def container(blob):
    """The pickle container as an `incoming.Container`, or None where the blob is not laid out as
    this module (or the reference on the same torch) writes it."""
    if _PREFIX is None:
        return None
    whole = hostmem.view(blob)
    try:
        out = _Reader(*_condense(blob), whole).load()
        cdf, k, v = out.cdf, out.max_tensors_key, out.max_tensors_value
        rows, C, lp = cdf.shape
        L, T = k.shape[:2]
        chunks = out.data_chunks
        maxima_types = (torch.float16, torch.bfloat16)
        fine = (rows == 2 * L and lp >= 2 and cdf.dtype is torch.int16 and out.num_heads * out.head_size == C and T > 0
                and k.dtype in maxima_types and v.dtype is k.dtype and v.shape[:2] == (L, T)
                and k.host.numel() == v.host.numel() == 2 * L * T and len(chunks) == -(-T // wire.MAX_STREAM_BYTES))
        for g, c in enumerate(chunks if fine else ()):
            fine = (fine and c.bytestream.dtype is torch.uint8 and c.bytestream_lengths.dtype is torch.int32
                    and c.bytestream_lengths.shape == (rows, C)
                    and c.ntokens == min(wire.MAX_STREAM_BYTES, T - g * wire.MAX_STREAM_BYTES))
    except (_NotPlain, AttributeError, TypeError, ValueError, KeyError, IndexError, struct.error):
        return None
    if not fine:
        return None
    c = Container(L, T, out.num_heads, out.head_size, T, lp - 1, 0, k.dtype is torch.bfloat16, False)
    c.tables = c.add(cdf.host)
    c.maxima = c.add(k.host)
    c.add(v.host, align=1)
    for i, chunk in enumerate(chunks):
        at = c.add(chunk.bytestream_lengths.host, align=64 if i == 0 else 1)
        if i == 0:
            c.lengths = at
        c.length_arrays.append((chunk.bytestream_lengths.host, 1))
    for i, chunk in enumerate(chunks):
        at = c.add(chunk.bytestream.host, align=64 if i == 0 else 1)
        if i == 0:
            c.payload = at
        c.payload_bytes += chunk.bytestream.host.numel()
    return c
