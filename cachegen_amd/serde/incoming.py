"""Containers on their way from host memory to decoded KV tensors.

A store hands back one blob per chunk.  All blobs of a call go to the GPU in one device buffer, as
they are (through pinned memory, in pieces, so that copying a piece on the host overlaps with the
bus carrying the piece before it), followed by an index that the host writes meanwhile: for every
sub-chunk where its tables, maxima, lengths, payload and output tokens are, and the running sums of
the stream lengths, which the host has to add up anyway to check them against the payload's size.
One launch then decodes every sub-chunk of every blob (`cg_decode_listed`): no per-blob launches,
no scan of the lengths on the device, no conversion of 16-bit lengths."""
import contextlib
import ctypes
import struct

import numpy as np
import torch

from .. import _lib, codec, hostmem
from . import wire

_ALIGN = 256
# Uploads of more than _WHOLE_BYTES have a stream of their own (_upload) and pass through a few pinned pieces.  Pieces
# cost the bus some 15 us each besides their bytes (42 MB merged from pieces of 4 MB 1338 us, of 8 MB 1250, of 8 MB with pinned
# memory for all of them 1225; a store of 59 MB is the same with either).
_WHOLE_BYTES = 16 << 20
_PIECE_BYTES, _PIECES = 8 << 20, 4
# Up to this, torch's own copies: the host, not the bus, is what such a call waits for, and what goes up by moves has to be
# kept until it is through.
_SMALL_BYTES = 1 << 20

_ITEM = struct.Struct("<10q4i")      # CgHostContainer
_SUB_BYTES = 96                      # sizeof(CgListedSub)


def _up(n, a=_ALIGN):
    return (n + a - 1) // a * a


class LengthsError(ValueError):
    """A container's stream lengths do not fit its payload."""


class Container:
    """One container in host memory: its geometry, and where its sections lie in an area of `size`
    bytes that `pieces` ((offset, uint8 host tensor), in order) fill."""

    def __init__(self, num_layers, num_tokens, num_heads, head_size, chunk_tokens, max_bins, delta_group, bf16_maxima, lengths_u16):
        self.num_layers, self.num_tokens, self.num_heads, self.head_size = num_layers, num_tokens, num_heads, head_size
        self.chunk_tokens, self.max_bins, self.delta_group = chunk_tokens, max_bins, delta_group
        self.bf16_maxima, self.lengths_u16 = bf16_maxima, lengths_u16
        self.pieces, self.size = [], 0
        self.tables = self.maxima = self.lengths = self.payload = self.payload_bytes = 0     # offsets in the area
        self.length_arrays = []          # (host tensor, sub-chunks) of the stream lengths
        self.symbols = None              # count tables: stored symbols per (chunk, row), uint8 on the host

    @classmethod
    def flat(cls, blob, header=None):
        """A blob of the flat container (either version); checks everything that the host can."""
        h = wire.read_header(blob) if header is None else header
        c = cls(h["num_layers"], h["num_tokens"], h["num_heads"], h["head_size"], h["chunk_tokens"], h["max_bins"],
                h["delta_group"], h["bf16_maxima"], h["lengths_u16"])
        geo = h["geometry"]
        whole = hostmem.view(blob)
        c.pieces, c.size = [(0, whole)], whole.numel()
        c.tables, c.maxima, c.lengths, c.payload = (geo[k][0] for k in ("cdf", "maxima", "lengths", "payload"))
        c.payload_bytes = h["payload_bytes"]
        c.length_arrays = [(whole[c.lengths:], h["nsub"])]
        if h["count_tables"]:
            c.symbols = wire.table_symbol_counts(blob, h)
        return c

    def add(self, host, align=64):
        """Appends a section's bytes to the area; returns their offset."""
        at = _up(self.size, align)
        self.pieces.append((at, host))
        self.size = at + host.numel()
        return at


_upload_streams = {}                 # one per device, kept for the process


def _upload(pieces, total, index_at, write_index):
    """Device buffer of `total` bytes holding the pieces ((offset, host tensor), in order) and, from
    index_at on, what write_index(device address, uint8 tensor in pinned memory) puts there;
    write_index runs while the pieces before it are on the bus.

    A large transfer has a stream of its own, which the current stream waits for: the blobs of a
    call are on the bus while what the caller queued before (as a rule the decode of the blobs before
    them) still runs (32 blobs of 54 MB in all, one call behind the other: 1.46 -> 1.28 ms).  The
    buffer comes from that stream's memory and goes back when the current stream is through with it.
    For a small one the events and the change of stream cost more than they hide (+25 us)."""
    device = torch.device("cuda", torch.cuda.current_device())          # the caller made it current
    if index_at <= _WHOLE_BYTES:
        return _transfer(pieces, total, index_at, write_index, device)
    side = _upload_streams.get(device.index)
    if side is None:
        side = _upload_streams.setdefault(device.index, torch.cuda.Stream(device))
    current = torch.cuda.current_stream()
    with torch.cuda.stream(side):
        buf = _transfer(pieces, total, index_at, write_index, device, current)
    buf.record_stream(current)
    return buf


def _transfer(pieces, total, index_at, write_index, device, waiting=None):
    """waiting: a stream that waits for everything."""
    buf = torch.empty(total, dtype=torch.uint8, device=device)
    base = buf.data_ptr()
    if total <= _SMALL_BYTES:
        for at, end, write in ((0, index_at, lambda host: [host[a:a + t.numel()].copy_(t) for a, t in pieces]),
                               (index_at, total, lambda host: write_index(base, host))):
            host = hostmem.pinned(end - at)
            write(host)
            buf[at:end].copy_(host, non_blocking=True)
        return buf
    through = hostmem.event(device)
    moves = hostmem.Moves(device, codec._stream(device))
    try:
        if index_at <= _WHOLE_BYTES:
            moves.stage(pieces, base, index_at, _PIECE_BYTES // 128 * 64)
        else:
            moves.stage(pieces, base, index_at, _PIECE_BYTES, _PIECES)
        host = hostmem.pinned(total - index_at)
        write_index(base, host)
        moves.up(host, base + index_at)
    finally:
        through.record()
        if waiting is not None:
            waiting.wait_event(through)                  # before `hold`: from then on the next call may record it again
        moves.hold(through)
    return buf


def _levels(bins, num_layers, device):
    """A bins vector as the kernels and the index take it: float32, dense, on `device`, or on the host
    if it is there."""
    if bins.numel() != num_layers:
        raise RuntimeError("bins vectors must have one entry per layer (%d), got %d" % (num_layers, bins.numel()))
    return bins.detach().to(device=device if bins.is_cuda else bins.device, dtype=torch.float32).reshape(-1).contiguous()


def decode(items, out, fmt):
    """Decodes containers into one tensor.  items: [(Container, key_bins, value_bins, t0)]: levels
    (tensors of L values, as `codec.decode_kv` takes them; those on the CPU travel with the index) and
    first output token of each; all containers have the same layers, heads and head size.  out: KV
    tensor in layout `fmt` on the GPU."""
    first = items[0][0]
    L, H, D = first.num_layers, first.num_heads, first.head_size
    C, rows, device = H * D, 2 * first.num_layers, out.device
    lib = _lib.lib()
    # everything that can be refused is, before anything is queued
    T = codec.check_output(out, L, H, D, fmt)
    # launches: containers that share a table length (and the delta grouping), side by side
    launches = {}
    for item in items:
        c = item[0]
        if (c.num_layers, c.num_heads, c.head_size) != (L, H, D):
            raise ValueError("containers of different caches in one call")
        if c.payload_bytes <= 0:
            raise RuntimeError("payload must be a contiguous, non-empty uint8 tensor")
        if item[3] < 0 or item[3] + c.num_tokens > T:
            raise RuntimeError("output tensor does not match the encoded geometry")
        launches.setdefault((c.max_bins, c.delta_group), []).append(item)
    # levels by their tensors (`items` holds these): one conversion and one place in the index for each
    levels = {id(t): t for _, kb, vb, _ in items for t in (kb, vb)}
    levels = {k: _levels(t, L, device) for k, t in levels.items()}
    # areas: containers, then the index: running sums, the sub-chunks' entries, what the count
    # tables are rebuilt from, levels that are still on the host
    pieces, pos, nsubs = [], 0, 0
    plan = []                                        # (launch, container, its place, its rebuilt tables' place)
    counted = {}                                     # launch -> (containers with count tables, rebuilt tables, groups)
    for key, members in launches.items():
        groups = 0
        for c, kb, vb, t_out in members:
            pieces += [(pos + off, src) for off, src in c.pieces]
            plan.append((key, c, kb, vb, t_out, pos, groups))
            pos = _up(pos + c.size)
            nsubs += sum(n for _, n in c.length_arrays)
            if c.symbols is not None:
                groups += c.symbols.size
        if groups:
            counted[key] = (torch.empty((groups, C, key[0] + 1), dtype=torch.int16, device=device), groups)
    index_at = pos
    subs_at = _up(nsubs * rows * -(-C // 64) * 4)
    size = subs_at + nsubs * _SUB_BYTES
    groups_at = {}
    for key, (_, groups) in counted.items():
        groups_at[key] = size = _up(size, 64)
        size += groups * 8 + groups * 4 + groups     # starts, tokens, symbols
    levels_at = {}                                   # levels that are still on the host -> offset in the index
    for k, t in levels.items():
        if not t.is_cuda:
            levels_at[k] = size = _up(size, 64)
            size += 4 * L
    total = index_at + size

    def write_index(base, host):
        raw = host.numpy()
        index = base + index_at
        for k, at in levels_at.items():
            raw[at:at + 4 * L].view(np.float32)[:] = levels[k].numpy()

        def address(t):
            return index + levels_at[id(t)] if id(t) in levels_at else levels[id(t)].data_ptr()
        described = bytearray(len(plan) * _ITEM.size)
        arrays, array_subs = [], []
        for i, (key, c, kb, vb, t_out, place, group) in enumerate(plan):
            tables = place + base + c.tables
            if c.symbols is not None:
                rebuilt, groups = counted[key]
                tables = rebuilt.data_ptr() + group * C * (key[0] + 1) * 2
                at, n = groups_at[key], c.symbols.size
                sizes = np.multiply(c.symbols, C, dtype=np.int64)
                raw[at + 8 * group:at + 8 * (group + n)].view(np.int64)[:] = place + c.tables + n + np.cumsum(sizes) - sizes
                tokens = wire.chunk_token_counts(c.num_tokens, c.chunk_tokens)
                raw[at + 8 * groups + 4 * group:at + 8 * groups + 4 * (group + n)].view(np.int32)[:] = \
                    tokens[0] if len(tokens) == 1 else np.repeat(np.asarray(tokens, dtype=np.int32), rows)
                raw[at + 12 * groups + group:at + 12 * groups + group + n] = c.symbols
            _ITEM.pack_into(described, i * _ITEM.size, tables, place + base + c.maxima, place + base + c.lengths,
                            place + base + c.payload, c.payload_bytes, address(kb), address(vb), t_out, c.num_tokens, c.chunk_tokens,
                            c.max_bins, _lib.DT_BF16 if c.bf16_maxima else _lib.DT_F16, int(c.lengths_u16), len(c.length_arrays))
            for lengths, n in c.length_arrays:
                arrays.append(lengths.data_ptr())
                array_subs.append(n)
        n = len(arrays)
        bad = ctypes.c_int(0)
        start = host.data_ptr()
        if lib.cg_host_list((ctypes.c_char * len(described)).from_buffer(described), len(plan), (ctypes.c_void_p * n)(*arrays),
                            (ctypes.c_int64 * n)(*array_subs), L, C, start, index, start + subs_at, ctypes.byref(bad)) != _lib.CG_OK:
            raise LengthsError("wire container: payload size is not the sum of the stream lengths")

    with torch.cuda.device(device):
        buf = _upload(pieces, total, index_at, write_index)
        base = buf.data_ptr() + index_at
        stream = codec._stream(buf.device)
        # a word that stays zero unless a kernel finds counts that make no table
        with hostmem.StoredWords(1, torch.int32) if counted else contextlib.nullcontext() as verdict:
            for key, (tables, groups) in counted.items():
                at = base + groups_at[key]
                _lib.check(lib.cg_rebuild_tables(buf.data_ptr(), index_at, key[0], groups, C, at + 8 * groups, at + 12 * groups, at,
                                                 tables.data_ptr(), verdict.words.data_ptr(), stream))
            if counted:
                verdict.stored(by=hostmem.Moves(device, stream).here())
            at = base + subs_at
            for key, members in launches.items():
                n = sum(k for c, _, _, _ in members for _, k in c.length_arrays)
                codec.decode_listed(at, n, key[0], L, H, D, key[1], out, fmt)
                at += n * _SUB_BYTES
            if counted and verdict.read()[0]:        # the tables are waited for, not the decode behind them
                raise ValueError("wire container: histogram counts do not add up to the chunk's tokens")
    return out
