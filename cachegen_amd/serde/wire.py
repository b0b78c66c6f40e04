"""Flat wire container for encoded KV chunks.

The reference ships a chunk as a pickle of `CacheGenGPUEncoderOutput` holding GPU tensors
(LMCache/lmcache/storage_backend/serde/cachegen_basics.py:110-122): one device-to-host copy
per tensor when it is written, code execution from the blob when it is read.  This container
carries the same fields in one flat, versioned, little-endian buffer.  To write it, the encoder's
tensors go to pinned memory as they are, and the blob is put together on the host; to read it, the
blob goes to the GPU whole and is decoded from there (`incoming`), and reading it executes nothing.
`CacheGenDeserializer.from_bytes` accepts both forms (it looks at the first four bytes); the pickle
form stays the default for drop-in use.

Layout (every section starts on a 64-byte boundary; the gaps are zero):

    header   64 bytes   see HEADER
    cdf      int16  [nchunks, 2L, C, max_bins + 1]
    maxima   16-bit [2, L, T]           (float16 or bfloat16 bit patterns, see flags)
    lengths  int32  [nsub, 2L, C]       bytes of every stream, in stream order
    payload  uint8  [payload_bytes]     all streams back to back

Stream offsets are not stored: they are the running sum of `lengths` (cachegen_decoder.py:70 adds
it up on the GPU; the reader here does so on the host, where it checks it against the payload's
size, and sends every 64th along with the blob).  A stream longer than 256
bytes is stored cut to 256 (its length field keeps the full value), as in the device format.

Version 2 ("compact") stores the same information in fewer bytes, for chunks of at most 256
tokens, where the 66-byte table per 256-symbol stream outweighs the payload:

    tables   nsym uint8 [nchunks, 2L]: symbols that occur in a (chunk, row), then for every
             (chunk, row, channel) the first nsym histogram counts as one byte each
    lengths  uint16 when every length fits

A table is a function of its histogram (cal_cdf.cu:29-49: cdf[i] = (0xFFFF - max_bins) *
cum[i] / n + i), and for n <= 256 tokens the histogram is recovered from the table exactly
(the scale exceeds n, so distinct running sums give distinct quotients); the writer checks that
the rebuilt tables equal the originals and keeps the raw tables otherwise.  A count of 256
(one symbol for a whole chunk) is stored as 255; the reader adds what is missing from the
chunk's token count back to that entry.
"""
import struct
from typing import Dict, List, Optional, Tuple

import numpy as np

MAGIC = b"CGKV"
VERSION = 1
VERSION_COMPACT = 2
ALIGN = 64
HEADER_BYTES = 64
# magic, version, flags, L, T, H, D, chunk_tokens, max_bins, delta_group, nsub, payload_bytes,
# tables_bytes (version 2 only; zero in version 1)
HEADER = struct.Struct("<4sHHIIIIIIIIQQ")
FLAG_BF16_MAXIMA = 1
FLAG_COUNT_TABLES = 2        # version 2: tables stored as histogram counts
FLAG_LENGTHS_U16 = 4         # version 2: lengths stored as uint16
MAX_STREAM_BYTES = 256


def _up(n: int) -> int:
    return (n + ALIGN - 1) // ALIGN * ALIGN


def is_flat(blob) -> bool:
    return len(blob) >= 4 and bytes(blob[:4]) == MAGIC


def geometry(num_layers: int, num_tokens: int, num_heads: int, head_size: int, chunk_tokens: int,
             max_bins: int, payload_bytes: int, tables_bytes: Optional[int] = None,
             lengths_itemsize: int = 4) -> Dict[str, Tuple[int, int]]:
    """Section name -> (byte offset, byte size), plus "total" -> (size of the blob, 0).
    tables_bytes: size of the table section when it does not hold raw tables."""
    if min(num_layers, num_tokens, num_heads, head_size, chunk_tokens, max_bins) <= 0 or payload_bytes < 0:
        raise ValueError("wire container: sizes must be positive")
    C = num_heads * head_size
    nchunks = -(-num_tokens // chunk_tokens)
    full, rest = divmod(num_tokens, chunk_tokens)
    nsub = full * (-(-chunk_tokens // MAX_STREAM_BYTES)) + (-(-rest // MAX_STREAM_BYTES))
    raw_tables = nchunks * 2 * num_layers * C * (max_bins + 1) * 2
    sizes = [("cdf", raw_tables if tables_bytes is None else tables_bytes),
             ("maxima", 2 * num_layers * num_tokens * 2),
             ("lengths", nsub * 2 * num_layers * C * lengths_itemsize),
             ("payload", payload_bytes)]
    out, pos = {}, HEADER_BYTES
    for name, size in sizes:
        out[name] = (pos, size)
        pos = _up(pos + size)
    out["total"] = (pos, 0)
    out["nsub"] = (nsub, 0)
    out["nchunks"] = (nchunks, 0)
    return out


def write_header(num_layers, num_tokens, num_heads, head_size, chunk_tokens, max_bins, delta_group,
                 nsub, payload_bytes, bf16_maxima, version=VERSION, extra_flags=0, tables_bytes=0) -> bytes:
    flags = (FLAG_BF16_MAXIMA if bf16_maxima else 0) | extra_flags
    head = HEADER.pack(MAGIC, version, flags, num_layers, num_tokens, num_heads, head_size, chunk_tokens,
                       max_bins, delta_group, nsub, payload_bytes, tables_bytes)
    return head + bytes(HEADER_BYTES - len(head))


def read_header(blob) -> dict:
    """Validates magic, version and sizes; raises ValueError on anything inconsistent."""
    if len(blob) < HEADER_BYTES:
        raise ValueError("wire container: shorter than its header")
    magic, version, flags, L, T, H, D, S, max_bins, delta_group, nsub, payload_bytes, tables_bytes = \
        HEADER.unpack_from(bytes(blob[:HEADER.size]))
    if magic != MAGIC:
        raise ValueError("wire container: bad magic %r" % magic)
    if version not in (VERSION, VERSION_COMPACT):
        raise ValueError("wire container: version %d is not supported (this reader: up to %d)"
                         % (version, VERSION_COMPACT))
    known = FLAG_BF16_MAXIMA if version == VERSION else FLAG_BF16_MAXIMA | FLAG_COUNT_TABLES | FLAG_LENGTHS_U16
    if flags & ~known:
        raise ValueError("wire container: unknown flags 0x%x" % flags)
    count_tables = bool(flags & FLAG_COUNT_TABLES)
    if count_tables and S > MAX_STREAM_BYTES:
        raise ValueError("wire container: count tables need chunks of at most 256 tokens")
    geo = geometry(L, T, H, D, S, max_bins, payload_bytes, tables_bytes if count_tables else None,
                   2 if flags & FLAG_LENGTHS_U16 else 4)
    if geo["nsub"][0] != nsub:
        raise ValueError("wire container: %d sub-chunks recorded, geometry gives %d" % (nsub, geo["nsub"][0]))
    if len(blob) != geo["total"][0]:
        raise ValueError("wire container: %d bytes, geometry gives %d" % (len(blob), geo["total"][0]))
    if payload_bytes > nsub * 2 * L * H * D * MAX_STREAM_BYTES:
        raise ValueError("wire container: payload larger than 256 bytes per stream")
    return dict(num_layers=L, num_tokens=T, num_heads=H, head_size=D, chunk_tokens=S, max_bins=max_bins,
                delta_group=delta_group, nsub=nsub, payload_bytes=payload_bytes,
                bf16_maxima=bool(flags & FLAG_BF16_MAXIMA), count_tables=count_tables,
                lengths_u16=bool(flags & FLAG_LENGTHS_U16), version=version, geometry=geo)


def table_symbol_counts(blob, h) -> np.ndarray:
    """Version 2 with count tables: the symbols stored per (chunk, row), uint8 [nchunks * 2L], checked
    against the table length and the size of the section."""
    groups = h["geometry"]["nchunks"][0] * 2 * h["num_layers"]
    off, size = h["geometry"]["cdf"]
    if size < groups:
        raise ValueError("wire container: table section does not match its symbol counts")
    nsym = np.frombuffer(blob, dtype=np.uint8, count=groups, offset=off)
    if int(nsym.min()) < 1 or int(nsym.max()) > h["max_bins"]:
        raise ValueError("wire container: symbol count outside the table")
    if groups + int(nsym.sum(dtype=np.int64)) * h["num_heads"] * h["head_size"] != size:
        raise ValueError("wire container: table section does not match its symbol counts")
    return nsym


# --------------------------------------------------------------------------- #
# tables <-> histogram counts (numpy: the definition; the device code below mirrors it)
# --------------------------------------------------------------------------- #
def chunk_token_counts(num_tokens: int, chunk_tokens: int) -> List[int]:
    return [min(chunk_tokens, num_tokens - t0) for t0 in range(0, num_tokens, chunk_tokens)]


def tables_to_counts(cdf: np.ndarray, tokens: List[int]) -> Optional[np.ndarray]:
    """cdf uint16 [nchunks, 2L, C, Lp] built over tokens[chunk] <= 256 tokens each ->
    histogram counts int64 [nchunks, 2L, C, Lp - 1], or None if the tables are not exactly what
    cal_cdf.cu:29-49 gives for some histogram."""
    lp = cdf.shape[-1]
    scale = 0xFFFF - (lp - 1)
    n = np.asarray(tokens, dtype=np.int64).reshape(-1, 1, 1, 1)
    q = cdf.astype(np.int64) - np.arange(lp, dtype=np.int64)
    cum = (q * n + scale - 1) // scale
    counts = np.diff(cum, axis=-1)
    if (cum[..., 0] != 0).any() or (counts < 0).any() or not np.array_equal(counts_to_tables(counts, tokens), cdf):
        return None
    return counts


def counts_to_tables(counts: np.ndarray, tokens: List[int]) -> np.ndarray:
    """The inverse: cdf[i] = (0xFFFF - max_bins) * cum[i] / n + i in integers."""
    lp = counts.shape[-1] + 1
    scale = 0xFFFF - (lp - 1)
    n = np.asarray(tokens, dtype=np.int64).reshape(-1, 1, 1, 1)
    cum = np.concatenate([np.zeros(counts.shape[:-1] + (1,), dtype=np.int64), np.cumsum(counts, axis=-1)], axis=-1)
    return ((scale * cum) // n + np.arange(lp, dtype=np.int64)).astype(np.uint16)


def pack_counts(counts: np.ndarray) -> Tuple[np.ndarray, np.ndarray]:
    """-> (nsym uint8 [nchunks, 2L], bytes uint8 [sum of C * nsym]): per (chunk, row) the number
    of leading symbols that hold every occurrence, then those counts, clamped to 255, for each
    channel in turn."""
    used = counts.sum(axis=2) > 0                                    # [nchunks, 2L, nsyms]
    nsyms = counts.shape[-1]
    nsym = np.where(used.any(-1), nsyms - np.argmax(used[..., ::-1], axis=-1), 1).astype(np.uint8)
    mask = np.arange(nsyms)[None, None, None, :] < nsym[:, :, None, None].astype(np.int64)
    mask = np.broadcast_to(mask, counts.shape)
    return nsym, np.minimum(counts, 255).astype(np.uint8)[mask]


def unpack_counts(nsym: np.ndarray, data: np.ndarray, C: int, nsyms: int, tokens: List[int]) -> np.ndarray:
    mask = np.arange(nsyms)[None, None, None, :] < nsym[:, :, None, None].astype(np.int64)
    mask = np.broadcast_to(mask, nsym.shape + (C, nsyms))
    if int(mask.sum()) != data.size:
        raise ValueError("wire container: table section does not match its symbol counts")
    counts = np.zeros(mask.shape, dtype=np.int64)
    counts[mask] = data
    n = np.asarray(tokens, dtype=np.int64).reshape(-1, 1, 1)
    missing = n - counts.sum(-1)                                     # 1 where a count of 256 was clamped
    if ((missing != 0) & ~((missing == 1) & ((counts == 255).sum(-1) == 1))).any():
        raise ValueError("wire container: histogram counts do not add up to the chunk's tokens")
    return counts + (counts == 255) * missing[..., None]


# --------------------------------------------------------------------------- #
# host form (numpy): the definition of the format, used by the CPU tests
# --------------------------------------------------------------------------- #
def pack_host(cdf: np.ndarray, maxima_bits: np.ndarray, lengths: np.ndarray, payload: np.ndarray,
              num_heads: int, head_size: int, chunk_tokens: int, delta_group: int = 0,
              bf16_maxima: bool = False, compact: bool = False) -> bytes:
    """cdf int16/uint16 [nchunks, 2L, C, Lp]; maxima_bits uint16 [2, L, T]; lengths int32
    [nsub, 2L, C]; payload uint8 [n].  compact: write version 2."""
    nchunks, rows, C, lp = cdf.shape
    L, T = maxima_bits.shape[1:]
    if rows != 2 * L or C != num_heads * head_size or lengths.shape[1:] != (rows, C):
        raise ValueError("wire container: array shapes do not agree")
    cdf = np.ascontiguousarray(cdf)
    if cdf.dtype == np.int16:
        cdf = cdf.view(np.uint16)
    version, flags, tables, lengths_out = VERSION, 0, cdf.astype("<u2", copy=False).tobytes(), lengths.astype("<i4")
    tables_bytes = None
    if compact:
        version = VERSION_COMPACT
        counts = tables_to_counts(cdf, chunk_token_counts(T, chunk_tokens)) if chunk_tokens <= MAX_STREAM_BYTES else None
        if counts is not None:
            nsym, data = pack_counts(counts)
            tables = nsym.tobytes() + data.tobytes()
            tables_bytes = len(tables)
            flags |= FLAG_COUNT_TABLES
        if lengths.size == 0 or (int(lengths.min()) >= 0 and int(lengths.max()) <= 0xFFFF):
            lengths_out = lengths.astype("<u2")
            flags |= FLAG_LENGTHS_U16
    geo = geometry(L, T, num_heads, head_size, chunk_tokens, lp - 1, payload.size, tables_bytes,
                   lengths_out.dtype.itemsize)
    if geo["nchunks"][0] != nchunks or geo["nsub"][0] != lengths.shape[0]:
        raise ValueError("wire container: chunk counts do not agree with the token count")
    if int(np.minimum(lengths, MAX_STREAM_BYTES).astype(np.int64).sum()) != payload.size:
        raise ValueError("wire container: payload size is not the sum of the stream lengths")
    buf = bytearray(geo["total"][0])
    buf[:HEADER_BYTES] = write_header(L, T, num_heads, head_size, chunk_tokens, lp - 1, delta_group,
                                      lengths.shape[0], payload.size, bf16_maxima, version, flags,
                                      tables_bytes or 0)
    for name, raw in (("cdf", tables), ("maxima", np.ascontiguousarray(maxima_bits).astype("<u2", copy=False).tobytes()),
                      ("lengths", np.ascontiguousarray(lengths_out).tobytes()),
                      ("payload", np.ascontiguousarray(payload).tobytes())):
        off, size = geo[name]
        assert len(raw) == size
        buf[off:off + size] = raw
    return bytes(buf)


def unpack_host(blob):
    """-> (header dict, cdf uint16 [nchunks, 2L, C, Lp], maxima uint16 [2, L, T], lengths int32
    [nsub, 2L, C], payload uint8 [n]): read-only numpy views of the blob where the stored form is
    the array itself, new arrays where it is not (version 2)."""
    h = read_header(blob)
    geo = h["geometry"]
    L, T, C = h["num_layers"], h["num_tokens"], h["num_heads"] * h["head_size"]
    lp, nchunks = h["max_bins"] + 1, geo["nchunks"][0]
    mv = memoryview(blob)

    def section(name, dt, shape):
        off, size = geo[name]
        return np.frombuffer(mv[off:off + size], dtype=dt).reshape(shape)
    if h["count_tables"]:
        raw = section("cdf", "u1", (-1,))
        if raw.size < nchunks * 2 * L:
            raise ValueError("wire container: table section does not match its symbol counts")
        nsym = raw[:nchunks * 2 * L].reshape(nchunks, 2 * L)
        if int(nsym.min()) < 1 or int(nsym.max()) > lp - 1:
            raise ValueError("wire container: symbol count outside the table")
        tokens = chunk_token_counts(T, h["chunk_tokens"])
        cdf = counts_to_tables(unpack_counts(nsym, raw[nchunks * 2 * L:], C, lp - 1, tokens), tokens)
    else:
        cdf = section("cdf", "<u2", (nchunks, 2 * L, C, lp))
    maxima = section("maxima", "<u2", (2, L, T))
    lengths = section("lengths", "<u2" if h["lengths_u16"] else "<i4", (h["nsub"], 2 * L, C)).astype(np.int32, copy=False)
    payload = section("payload", "u1", (h["payload_bytes"],))
    if int(np.minimum(lengths, MAX_STREAM_BYTES).astype(np.int64).sum()) != h["payload_bytes"] \
            or (lengths.size and int(lengths.min()) < 0):
        raise ValueError("wire container: payload size is not the sum of the stream lengths")
    return h, cdf, maxima, lengths, payload


# --------------------------------------------------------------------------- #
# device form: out of the encoder's tensors
# --------------------------------------------------------------------------- #
def _device_counts_launch(cdf, tokens):
    """Device form of tables_to_counts for cdf int16 [nchunks, 2L, C, Lp]: launches the conversion
    and returns (dense counts uint8 [G, C, Lp-1], nsym int32 [G], inexact int32 [1]), all still on
    the device and not waited for.  tokens: per chunk; all but the last are the same."""
    import torch
    from .. import _lib, codec
    nchunks, rows, C, lp = cdf.shape
    G = nchunks * rows
    dev = cdf.device
    cdf = cdf.contiguous()
    tok = torch.full((G,), tokens[0], dtype=torch.int32, device=dev)
    if tokens[-1] != tokens[0]:
        tok[G - rows:].fill_(tokens[-1])
    dense = torch.empty((G, C, lp - 1), dtype=torch.uint8, device=dev)
    nsym = torch.empty(G, dtype=torch.int32, device=dev)
    inexact = torch.empty(1, dtype=torch.int32, device=dev)
    with torch.cuda.device(dev):
        _lib.check(_lib.lib().cg_tables_to_counts(cdf.data_ptr(), lp - 1, G, C, tok.data_ptr(), dense.data_ptr(),
                                                  nsym.data_ptr(), inexact.data_ptr(), codec._stream(dev)))
    return dense, nsym, inexact


def _device_tables(nsym_host, nsym_dev, data, C, lp, tokens):
    """Device form of unpack_counts + counts_to_tables -> cdf int16 [nchunks, 2L, C, Lp].
    nsym_host: numpy uint8 [nchunks, 2L] (read from the blob on the host), nsym_dev the same bytes
    on the device."""
    import torch
    from .. import _lib, codec
    nchunks, rows = nsym_host.shape
    G = nchunks * rows
    dev = data.device
    sizes = nsym_host.astype(np.int64).ravel() * C
    starts = np.concatenate([[0], np.cumsum(sizes)[:-1]]).astype(np.int64)
    if int(sizes.sum()) != data.numel():
        raise ValueError("wire container: table section does not match its symbol counts")
    small = torch.from_numpy(np.concatenate([starts, np.repeat(np.asarray(tokens, dtype=np.int64), rows)])).to(dev)
    tok = small[G:].to(torch.int32)
    cdf = torch.empty((nchunks, rows, C, lp), dtype=torch.int16, device=dev)
    invalid = torch.empty(1, dtype=torch.int32, device=dev)
    with torch.cuda.device(dev):
        _lib.check(_lib.lib().cg_counts_to_tables(data.data_ptr(), data.numel(), lp - 1, G, C, tok.data_ptr(),
                                                  nsym_dev.data_ptr(), small.data_ptr(), cdf.data_ptr(),
                                                  invalid.data_ptr(), codec._stream(dev)))
    if int(invalid.item()):
        raise ValueError("wire container: histogram counts do not add up to the chunk's tokens")
    return cdf


# Bytes of blobs that leave the GPU in one go: while the host copies one piece into its blobs, the
# next is on the bus.  Blobs of one 256-token chunk (6 MB) are a piece each; where that is all
# there is, long tables are cut in slices so that their copy overlaps with the rest's transfer (each
# transfer costs 6 to 15 us by itself: tables of 4.3 MB in two, one chunk to bytes and back 558 us, in one 544).
_PIECE_BYTES = 4 << 20
_SLICE_BYTES = 4 << 20


class HostPart:
    """Chunks [first, last) of an encoded tensor on their way to (pinned) host memory, one blob's
    worth: uint8 tensors `tables`, `lengths`, `payload` as they lie on the device, `maxima` (uint16
    numpy view [2L, tokens]), `sub_bytes` (payload bytes per sub-chunk), tokens [t0, t1).  `symbols`:
    stored symbols per (chunk, row) where `tables` holds histogram counts, else None;
    `lengths_itemsize` 2 or 4.  Sizes are known and the maxima are there from the start; the other
    bytes are there after `arrive`."""

    def arrive(self):
        """Waits for everything."""
        self.arrived.synchronize()

    def fill(self, parts):
        """[(uint8 tensor in ordinary memory, slice of `tables`, `lengths` or `payload`, its arrival)]: copied as they
        arrive."""
        self.moves.fill(parts)


def bring_to_host(enc, first_chunk, num_chunks, per_chunk=True, compact=False):
    """Yields a HostPart per chunk (or one for all of them) once its sizes are known.

    The sections leave the encoder's own tensors for pinned memory as they are; blobs are put
    together on the host, where they have to be written anyway: no second copy of them on the
    device.  The host waits for the device once for the sizes (status, payload offsets, symbol
    counts, stored into pinned memory by one kernel) and the maxima while the tables, whose size it
    knows, are already on the bus, and then for each piece of about _PIECE_BYTES."""
    import torch
    from .. import codec, hostmem
    dev = enc.payload.device
    with torch.cuda.device(dev):
        moves = hostmem.Moves(dev, codec._stream(dev))
    with moves:
        yield from _bring_to_host(enc, first_chunk, num_chunks, per_chunk, compact, moves)


def _bring_to_host(enc, first_chunk, num_chunks, per_chunk, compact, moves):
    import torch
    from .. import _lib, hostmem
    L, H, D, S, T = enc.num_layers, enc.num_heads, enc.head_size, enc.chunk_tokens, enc.num_tokens
    C = H * D
    rows = 2 * L
    spc = enc.subchunks_per_chunk
    c_first, c_last = first_chunk, first_chunk + num_chunks
    g_first, g_last = c_first * spc, min(c_last * spc, enc.lengths.shape[0])
    tokens = chunk_token_counts(T, S)[c_first:c_last]
    dev = enc.payload.device
    lib = _lib.lib()

    def fetch_tables(src):
        """(pinned tables, [(end, arrival)]): in slices where nothing else would overlap with them."""
        n = src.numel() * src.element_size()
        if len(pieces) > 1 or n < 2 * _SLICE_BYTES:
            host, arrival = moves.down(src)
            return host, [(n, arrival)]
        src, host = moves.room(src)
        ends = [n * (i + 1) // (n // _SLICE_BYTES) // 64 * 64 for i in range(n // _SLICE_BYTES - 1)] + [n]
        slices = []
        for at, end in zip([0] + ends, ends):
            slices.append((end, moves.down_to(src.data_ptr() + at, host[at:end])))
        return host, slices

    def subs(c):
        return min(c * spc, g_last) - g_first

    # blobs by pieces: (first blob, last blob) covering about _PIECE_BYTES of tables and lengths
    groups = [(c, c + 1) for c in range(c_first, c_last)] if per_chunk else [(c_first, c_last)]
    early = {}                                           # the first piece's tables and lengths: sizes not needed
    stream = moves.stream
    with torch.cuda.device(dev):
        cdf = enc.cdf[c_first:c_last]
        lengths = enc.lengths[g_first:g_last]
        wide = inexact = nsym = dense = None
        if compact:
            lengths16 = torch.empty(lengths.shape, dtype=torch.int16, device=dev)
            wide = torch.empty(1, dtype=torch.int32, device=dev)
            _lib.check(lib.cg_lengths_to_u16(lengths.data_ptr(), lengths.numel(), lengths16.data_ptr(), wide.data_ptr(), stream))
            if S <= MAX_STREAM_BYTES:
                dense, nsym, inexact = _device_counts_launch(cdf, tokens)
        nbounds, ngroups = g_last - g_first + 1, 0 if nsym is None else nsym.numel()

        def ptr(t):
            return None if t is None else t.data_ptr()
        with hostmem.StoredWords(3 + nbounds + ngroups, torch.int64) as words:
            _lib.check(lib.cg_wire_meta(enc.status.data_ptr(), enc.offsets[g_first * rows * C:].data_ptr(), rows * C, nbounds,
                                        ptr(wide), ptr(inexact), ptr(nsym), ngroups, words.words.data_ptr(), stream))
            chunk_bytes = max(1, cdf[0].numel() * cdf.element_size() + min(spc, lengths.shape[0]) * rows * C * 4)
            step = max(1, _PIECE_BYTES // chunk_bytes) if per_chunk else 1
            pieces = [(i, min(i + step, len(groups))) for i in range(0, len(groups), step)]
            tables_src, lengths_src = cdf, lengths
            if dense is not None:
                # ragged count bytes; their places follow from nsym, which is on the device
                tables_src = torch.empty(dense.numel(), dtype=torch.uint8, device=dev)
                _lib.check(lib.cg_pack_counts(dense.data_ptr(), dense.shape[2], ngroups, C, nsym.data_ptr(), None,
                                              tables_src.data_ptr(), stream))
            # behind the launches: a copy between two of them costs 20 us
            maxima, arrival = moves.down(enc.maxima)
            words.stored(by=arrival)                     # one wait for the words and the maxima
            if dense is None and not compact:
                a, b = groups[0][0], groups[pieces[0][1] - 1][1]
                early = {"tables": fetch_tables(cdf[a - c_first:b - c_first]), "lengths": moves.down(lengths[subs(a):subs(b)], place=False)}
            meta = words.read()

    enc.raise_for_status(meta[0])
    bounds = meta[3:3 + nbounds]
    symbols = starts = None                              # starts: byte offset of every chunk's counts in tables_src
    if compact:
        if dense is not None:
            if meta[2]:
                tables_src = cdf                         # not the tables of histograms: stored as they are
            else:
                symbols = np.asarray(meta[3 + nbounds:], dtype=np.uint8)
                starts = [0] + np.cumsum(symbols.reshape(-1, rows).sum(axis=1, dtype=np.int64) * C).tolist()
        if not meta[1]:
            lengths_src = lengths16                      # bit pattern of the uint16 value

    def table_range(a, b):
        if starts is not None:
            return tables_src[starts[a - c_first]:starts[b - c_first]]
        return tables_src[a - c_first:b - c_first]

    def queue(piece):
        a, b = groups[piece[0]][0], groups[piece[1] - 1][1]
        p0, p1 = bounds[subs(a)], bounds[subs(b)]
        with torch.cuda.device(dev):
            tables = early.pop("tables", None)
            lens = early.pop("lengths", None)
            return (fetch_tables(table_range(a, b)) if tables is None else tables,
                    moves.down(lengths_src[subs(a):subs(b)], place=False) if lens is None else lens, moves.down(enc.payload[p0:p1]))

    itemsize = lengths_src.element_size()
    queued = queue(pieces[0])
    for k, piece in enumerate(pieces):
        ((tables, slices), (lens, lens_arrived), (payload, arrived)), queued = queued, queue(pieces[k + 1]) if k + 1 < len(pieces) else None
        at = [0, 0, 0]
        for a, b in groups[piece[0]:piece[1]]:
            part = HostPart()
            part.first, part.last = a, b
            part.t0, part.t1 = a * S, min(b * S, T)
            part.sub_bytes = [bounds[g + 1] - bounds[g] for g in range(subs(a), subs(b))]
            n = [(starts[b - c_first] - starts[a - c_first]) if starts is not None else (b - a) * cdf[0].numel() * 2,
                 len(part.sub_bytes) * rows * C * itemsize, sum(part.sub_bytes)]
            part.tables, part.lengths, part.payload = (t[i:i + j] for t, i, j in zip((tables, lens, payload), at, n))
            at = [i + j for i, j in zip(at, n)]
            part.maxima = maxima.numpy().view(np.uint16).reshape(rows, T)[:, part.t0:part.t1]
            part.symbols = None if symbols is None else symbols[(a - c_first) * rows:(b - c_first) * rows]
            part.lengths_itemsize = itemsize
            part.moves, part.lengths_arrived, part.arrived = moves, lens_arrived, arrived
            # several blobs in a piece: all of the piece's tables, there with its last slice
            part.slices = slices if piece[1] - piece[0] == 1 else [(n[0], slices[-1][1])]
            yield part


def pack_chunks(enc, first_chunk: int = 0, num_chunks: Optional[int] = None, per_chunk: bool = True,
                compact: bool = False) -> List[bytes]:
    """Blobs for chunks [first_chunk, first_chunk + num_chunks) of an `EncodedKV`: one blob per
    chunk (what one `to_bytes` call of the reference covers) or, with per_chunk=False, a single
    blob holding all of them; compact: version 2."""
    import torch
    from .. import hostmem
    nch = enc.num_chunks
    if num_chunks is None:
        num_chunks = nch - first_chunk
    if first_chunk < 0 or num_chunks <= 0 or first_chunk + num_chunks > nch:
        raise ValueError("chunk range outside the encoded tensor")
    L, H, D = enc.num_layers, enc.num_heads, enc.head_size
    bf16 = enc.maxima.dtype == torch.bfloat16
    blobs = []
    for part in bring_to_host(enc, first_chunk, num_chunks, per_chunk, compact):
        T = part.t1 - part.t0
        nbytes = part.payload.numel()
        flags, tables_bytes = 0, None
        if part.symbols is not None:
            flags |= FLAG_COUNT_TABLES
            tables_bytes = part.symbols.size + part.tables.numel()
        if part.lengths_itemsize == 2:
            flags |= FLAG_LENGTHS_U16
        table_tokens = min(enc.chunk_tokens, T)          # a short last chunk is a blob of its own length
        geo = geometry(L, T, H, D, table_tokens, enc.max_bins, nbytes, tables_bytes, part.lengths_itemsize)
        head = write_header(L, T, H, D, table_tokens, enc.max_bins, enc.delta_group, len(part.sub_bytes), nbytes, bf16,
                            VERSION_COMPACT if compact else VERSION, flags, tables_bytes or 0)
        if part.symbols is not None:
            head += part.symbols.tobytes()
        blob, into = hostmem.new_bytes(geo["total"][0])
        raw, parts = into.numpy(), []
        end = len(head)
        raw[:end] = np.frombuffer(head, dtype=np.uint8)
        for section, src in (("cdf", part.tables), ("maxima", part.maxima), ("lengths", part.lengths), ("payload", part.payload)):
            off, size = geo[section]
            start = max(off, end)                        # count tables: the symbol counts are there already
            raw[end:start] = 0                           # the gap before the section
            end = off + size
            if section == "cdf":
                at = 0
                for e, arrival in part.slices:
                    parts.append((into[start + at:start + e], src[at:e], arrival))
                    at = e
            elif section == "maxima":
                np.copyto(raw[start:end].view(np.uint16).reshape(2 * L, T), src)
            else:
                parts.append((into[start:end], src, part.lengths_arrived if section == "lengths" else part.arrived))
        raw[end:] = 0
        part.fill(parts)
        blobs.append(blob)
    return blobs


def unpack_to_device(blob, device):
    """-> (header dict, cdf, maxima, lengths, payload) on the device, which the blob reached in a
    single copy from pinned host memory: views of that buffer where the stored form is the
    tensor itself, rebuilt tensors where it is not (version 2).  The stream lengths are checked
    against the payload size on the host.  For programs that want the sections themselves: the
    deserializer and the engine decode blobs without these tensors (incoming.py)."""
    import torch
    h = read_header(blob)
    geo = h["geometry"]
    L, T, C = h["num_layers"], h["num_tokens"], h["num_heads"] * h["head_size"]
    lp, nchunks = h["max_bins"] + 1, geo["nchunks"][0]
    from .. import hostmem
    host = hostmem.pinned(len(blob))
    host.copy_(hostmem.view(blob))
    buf = host.to(device, non_blocking=False)      # waits: the pinned buffer is free for the next call at once
    # the lengths are in the blob: their sum is checked here, without asking the device
    off, size = geo["lengths"]
    host_lengths = np.frombuffer(blob, dtype=np.uint16 if h["lengths_u16"] else np.int32, count=h["nsub"] * 2 * L * C,
                                 offset=off)
    # one rule everywhere: a stream occupies min(length, 256) bytes of the payload
    if int(np.minimum(host_lengths, MAX_STREAM_BYTES).sum(dtype=np.int64)) != h["payload_bytes"] \
            or (host_lengths.size and int(host_lengths.min()) < 0):
        raise ValueError("wire container: payload size is not the sum of the stream lengths")
    def section(name, dtype, shape):
        off, size = geo[name]
        return buf[off:off + size].view(dtype).view(shape)
    if h["count_tables"]:
        nsym_host = table_symbol_counts(blob, h).reshape(nchunks, 2 * L)
        raw = section("cdf", torch.uint8, (-1,))
        cdf = _device_tables(nsym_host, raw[:nchunks * 2 * L], raw[nchunks * 2 * L:], C, lp,
                             chunk_token_counts(T, h["chunk_tokens"]))
    else:
        cdf = section("cdf", torch.int16, (nchunks, 2 * L, C, lp))
    maxima = section("maxima", torch.bfloat16 if h["bf16_maxima"] else torch.float16, (2, L, T))
    if h["lengths_u16"]:
        lengths = section("lengths", torch.int16, (h["nsub"], 2 * L, C)).to(torch.int32) & 0xFFFF
    else:
        lengths = section("lengths", torch.int32, (h["nsub"], 2 * L, C))
    payload = section("payload", torch.uint8, (h["payload_bytes"],))
    return h, cdf, maxima, lengths, payload
