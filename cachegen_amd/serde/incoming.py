"""Containers on their way from host memory to decoded KV tensors.

A store hands back one blob per chunk.  All blobs of a call go to the GPU in one device buffer, as
they are (through pinned memory, in pieces, so that copying a piece on the host overlaps with the
bus carrying the piece before it), followed by an index that the host writes meanwhile: for every
sub-chunk where its tables, maxima, lengths, payload and output tokens are, and the running sums of
the stream lengths, which the host has to add up anyway to check them against the payload's size.
One launch then decodes every sub-chunk of every blob (`cg_decode_listed`): no per-blob launches,
no scan of the lengths on the device, no conversion of 16-bit lengths."""
import numpy as np
import torch

from .. import _lib, codec, hostmem
from . import wire

_ALIGN = 256
# Uploads of more than _WHOLE_BYTES are cut into pieces of _PIECE_BYTES: below it, one host copy
# and one transfer are faster than several of each (6 MB: 135 us whole, 151 in pieces of 4 MB),
# above it the overlap pays (54 MB: 1.51 ms whole, 1.25 in pieces).
_WHOLE_BYTES = 16 << 20
_PIECE_BYTES = 4 << 20

_SUB = np.dtype([("cdf", "<i8"), ("maxima", "<i8"), ("lengths", "<i8"), ("bytes", "<i8"), ("last_word", "<i8"), ("first", "<i8"),
                 ("tile_starts", "<i8"), ("key_bins", "<i8"), ("value_bins", "<i8"), ("t_out", "<i8"),
                 ("n", "<i4"), ("maxima_pitch", "<i4"), ("max_dt", "<i4"), ("lengths_u16", "<i4")])      # CgListedSub


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

    def tile_starts(self, into: np.ndarray, sub_bytes: np.ndarray) -> None:
        """Fills the running sums (uint32, see CgListedSub) and the bytes of every sub-chunk;
        raises ValueError if the lengths do not fit the payload."""
        rows, C = 2 * self.num_layers, self.num_heads * self.head_size
        per_sub = rows * -(-C // 64)
        at = 0
        for lengths, nsub in self.length_arrays:
            rc = _lib.lib().cg_host_tile_starts(lengths.data_ptr(), 2 if self.lengths_u16 else 4, nsub, rows, C,
                                                into[at * per_sub:].ctypes.data, sub_bytes[at:].ctypes.data)
            if rc != _lib.CG_OK:
                raise LengthsError("wire container: payload size is not the sum of the stream lengths")
            at += nsub
        if int(sub_bytes.sum()) != self.payload_bytes:
            raise LengthsError("wire container: payload size is not the sum of the stream lengths")


def _upload(pieces, total, index_at, write_index, device):
    """Device buffer of `total` bytes holding the pieces ((offset, host tensor), in order) and, from
    index_at on, what write_index(device address, uint8 tensor in pinned memory) puts there;
    write_index runs while the pieces before it are on the bus."""
    buf = torch.empty(total, dtype=torch.uint8, device=device)
    step = index_at if index_at <= _WHOLE_BYTES else _PIECE_BYTES
    k = 0
    for p0 in range(0, index_at, step):
        p1 = min(p0 + step, index_at)
        # pinned blocks come from and go back to torch's pool, which reuses one only when the copy
        # out of it is through
        host = torch.empty(p1 - p0, dtype=torch.uint8, pin_memory=True)
        while k < len(pieces) and pieces[k][0] < p1:
            off, src = pieces[k]
            a, b = max(off, p0), min(off + src.numel(), p1)
            host[a - p0:b - p0].copy_(src[a - off:b - off])
            if off + src.numel() > p1:
                break
            k += 1
        buf[p0:p1].copy_(host, non_blocking=True)
    host = torch.empty(total - index_at, dtype=torch.uint8, pin_memory=True)
    write_index(buf.data_ptr(), host)
    buf[index_at:].copy_(host, non_blocking=True)
    return buf


def decode(items, out, fmt):
    """Decodes containers into one tensor.  items: [(Container, key_bins, value_bins, t0)]: levels
    (float32 [L] tensors on the output's device, or on the CPU: these travel with the index) and
    first output token of each; all containers have the same layers, heads and head size.  out: KV
    tensor in layout `fmt` on the GPU."""
    first = items[0][0]
    L, H, D = first.num_layers, first.num_heads, first.head_size
    C, rows, device = H * D, 2 * first.num_layers, out.device
    tiles = -(-C // 64)
    if any((c.num_layers, c.num_heads, c.head_size) != (L, H, D) for c, _, _, _ in items):
        raise ValueError("containers of different caches in one call")
    # areas: containers, then per container its running sums, then the sub-chunks' entries, then
    # what the count tables are rebuilt from
    pieces, pos = [], 0
    places = []
    for c, _, _, _ in items:
        if c.payload_bytes <= 0:
            raise RuntimeError("payload must be a contiguous, non-empty uint8 tensor")
        places.append(pos)
        pieces += [(pos + off, src) for off, src in c.pieces]
        pos = _up(pos + c.size)
    index_at = pos
    # launches: containers that share a table length (and the delta grouping)
    launches = {}
    for i, (c, _, _, _) in enumerate(items):
        launches.setdefault((c.max_bins, c.delta_group), []).append(i)
    nsubs = [sum(n for _, n in c.length_arrays) for c, _, _, _ in items]
    starts_at, size = [], 0
    for n in nsubs:
        starts_at.append(size)
        size += n * rows * tiles * 4
    subs_at = size = _up(size)
    size += sum(nsubs) * _SUB.itemsize
    counted = {}                                     # launch -> (containers with count tables, rebuilt tables, index offsets)
    for key, members in launches.items():
        who = [i for i in members if items[i][0].symbols is not None]
        if who:
            G = sum(items[i][0].symbols.size for i in who)
            at = _up(size)
            counted[key] = (who, torch.empty((G, C, key[0] + 1), dtype=torch.int16, device=device), G, at)
            size = at + _up(G * 8) + _up(G * 4) + G                  # starts, tokens, symbols
    levels_at = {}                                   # levels that are still on the host -> offset in the index
    for _, kb, vb, _ in items:
        for t in (kb, vb):
            if t.numel() != L or t.dtype != torch.float32:
                raise RuntimeError("bins vectors must be float32 with one entry per layer (%d)" % L)
            if not t.is_cuda and id(t) not in levels_at:
                levels_at[id(t)] = (_up(size, 64), t)
                size = _up(size, 64) + 4 * L
    total = index_at + size

    def write_index(base, host):
        raw = host.numpy()
        subs = raw[subs_at:subs_at + sum(nsubs) * _SUB.itemsize].view(_SUB)
        rebuilt = {}
        for key, (who, tables, G, at) in counted.items():
            start = np.empty(G, dtype=np.int64)
            tokens = np.empty(G, dtype=np.int32)
            symbols = np.empty(G, dtype=np.uint8)
            g = 0
            for i in who:
                c = items[i][0]
                n = c.symbols.size
                sizes = c.symbols.astype(np.int64) * C
                start[g:g + n] = places[i] + c.tables + n + np.cumsum(sizes) - sizes
                tokens[g:g + n] = np.repeat(np.asarray(wire.chunk_token_counts(c.num_tokens, c.chunk_tokens), dtype=np.int32), rows)
                symbols[g:g + n] = c.symbols
                rebuilt[i] = tables.data_ptr() + g * C * (key[0] + 1) * 2
                g += n
            raw[at:at + 8 * G].view(np.int64)[:] = start
            raw[at + _up(8 * G):at + _up(8 * G) + 4 * G].view(np.int32)[:] = tokens
            raw[at + _up(8 * G) + _up(4 * G):][:G] = symbols
        for at, t in levels_at.values():
            raw[at:at + 4 * L].view(np.float32)[:] = t.numpy()

        def levels(t):
            return t.data_ptr() if t.is_cuda else base + index_at + levels_at[id(t)][0]
        at = 0
        for members in launches.values():
            for i in members:
                c, kb, vb, t_out = items[i]
                n, place = nsubs[i], base + places[i]
                per = rows * tiles
                sub_bytes = np.empty(n, dtype=np.int64)
                c.tile_starts(raw[starts_at[i]:starts_at[i] + n * per * 4].view(np.uint32), sub_bytes)
                e = subs[at:at + n]
                at += n
                g = np.arange(n)
                nsc = -(-c.chunk_tokens // wire.MAX_STREAM_BYTES)
                chunk = g // nsc
                t0 = chunk * c.chunk_tokens + (g - chunk * nsc) * wire.MAX_STREAM_BYTES
                tables = rebuilt.get(i, place + c.tables)
                e["cdf"] = tables + chunk * (rows * C * (c.max_bins + 1) * 2)
                e["maxima"] = place + c.maxima + t0 * 2
                e["lengths"] = place + c.lengths + g * (rows * C * (2 if c.lengths_u16 else 4))
                skew = (place + c.payload) & 3
                e["bytes"] = place + c.payload - skew
                e["last_word"] = (skew + c.payload_bytes - 1) & ~3
                e["first"] = skew + np.cumsum(sub_bytes) - sub_bytes
                e["tile_starts"] = base + index_at + starts_at[i] + g * (per * 4)
                e["key_bins"] = levels(kb)
                e["value_bins"] = levels(vb)
                e["t_out"] = t_out + t0
                e["n"] = np.minimum(np.minimum((chunk + 1) * c.chunk_tokens, c.num_tokens) - t0, wire.MAX_STREAM_BYTES)
                e["maxima_pitch"] = c.num_tokens
                e["max_dt"] = _lib.DT_BF16 if c.bf16_maxima else _lib.DT_F16
                e["lengths_u16"] = c.lengths_u16

    with torch.cuda.device(device):
        buf = _upload(pieces, total, index_at, write_index, device)
        base = buf.data_ptr() + index_at
        verdicts = []
        for key, (who, tables, G, at) in counted.items():
            invalid = torch.empty(1, dtype=torch.int32, device=device)
            _lib.check(_lib.lib().cg_counts_to_tables(
                buf.data_ptr(), index_at, key[0], G, C, base + at + _up(8 * G), base + at + _up(8 * G) + _up(4 * G), base + at,
                tables.data_ptr(), invalid.data_ptr(), codec._stream(buf.device)))
            verdict = torch.empty(1, dtype=torch.int32, pin_memory=True)
            verdict.copy_(invalid, non_blocking=True)
            verdicts.append(verdict)
        if verdicts:
            tables_done = torch.cuda.Event()
            tables_done.record()
        at = base + subs_at
        for key, members in launches.items():
            n = sum(nsubs[i] for i in members)
            codec.decode_listed(at, n, key[0], L, H, D, key[1], out, fmt)
            at += n * _SUB.itemsize
        if verdicts:
            tables_done.synchronize()                # the tables, not the decode behind them
            if any(int(v[0]) for v in verdicts):
                raise ValueError("wire container: histogram counts do not add up to the chunk's tokens")
    return out
