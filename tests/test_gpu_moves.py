"""Bytes between pinned and device memory, and what says how far a stream is."""
import threading

import pytest
import torch

from cachegen_amd import _lib, codec, hostmem

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda:0")
GUARD = 64


def _bytes(n, seed):
    return torch.randint(0, 256, (n,), generator=torch.Generator().manual_seed(seed), dtype=torch.uint8)


# one byte, either side of a 16-byte unit, of a block's 4 KB, of the launch's 256 KB, several of its rounds
@pytest.mark.parametrize("n", [1, 15, 16, 17, 4095, 4097, (256 << 10) - 1, (256 << 10) + 33, (3 << 20) + 5])
@pytest.mark.parametrize("at_host,at_dev", [(0, 0), (5, 5), (0, 1), (13, 2)])
def test_bytes_arrive_and_no_others_change(n, at_host, at_dev):
    print(n, at_host, at_dev, flush=True)
    want = _bytes(n, n)
    host = torch.full((n + at_host + GUARD,), 7, dtype=torch.uint8).pin_memory()
    back = torch.full((n + at_host + GUARD,), 9, dtype=torch.uint8).pin_memory()
    dev = torch.full((n + at_dev + GUARD,), 8, dtype=torch.uint8, device=DEV)
    host[at_host:at_host + n] = want
    with torch.cuda.device(DEV), hostmem.Moves(DEV, codec._stream(DEV)) as moves:
        moves.up(host[at_host:at_host + n], dev.data_ptr() + at_dev)
        arrival = moves.down_to(dev.data_ptr() + at_dev, back[at_host:at_host + n])
        arrival.synchronize()
        assert torch.equal(back[at_host:at_host + n], want)
    got = dev.cpu()
    assert torch.equal(got[at_dev:at_dev + n], want)
    assert (got[:at_dev] == 8).all() and (got[at_dev + n:] == 8).all()
    assert (back[:at_host] == 9).all() and (back[at_host + n:] == 9).all()


def test_arrivals_come_in_order_and_memory_is_kept():
    src = torch.arange(1 << 20, dtype=torch.int32, device=DEV)
    with torch.cuda.device(DEV), hostmem.Moves(DEV, codec._stream(DEV)) as moves:
        parts = [moves.down(src[i << 18:(i + 1) << 18]) for i in range(4)]
        for i in (2, 0, 3, 1):
            parts[i][1].synchronize()
            assert torch.equal(parts[i][0].view(torch.int32), torch.arange(i << 18, (i + 1) << 18, dtype=torch.int32))
        lost = moves.down(src)[1]                        # its memory is dropped here and kept by `moves`
    lost.synchronize()
    empty, arrival = hostmem.Moves(DEV, codec._stream(DEV)).down(src[:0])
    assert empty.numel() == 0


def test_memory_that_has_been_read_is_given_back(monkeypatch):
    monkeypatch.setattr(hostmem, "_HELD_BYTES", 1 << 20)
    dst = torch.empty(1 << 20, dtype=torch.uint8, device=DEV)
    for i in range(8):
        moves = hostmem.Moves(DEV, codec._stream(DEV))
        moves.up(_bytes(1 << 20, i).pin_memory(), dst.data_ptr())
        event = hostmem.event(DEV)
        event.record()
        moves.hold(event)
        assert sum(t.numel() for _, _, tensors in hostmem._held for t in tensors) <= 2 << 20       # the last one's, and the one it came on top of
    torch.cuda.synchronize()
    hostmem.event(DEV)
    assert not hostmem._held and len(hostmem._events[0]) <= 16
    assert torch.equal(dst.cpu(), _bytes(1 << 20, 7))


def test_marks_are_refused_where_they_cannot_be_set():
    lib = _lib.lib()
    word = torch.zeros(2, dtype=torch.int32).pin_memory()
    with pytest.raises(RuntimeError, match="misaligned"):
        _lib.check(lib.cg_mark(word.data_ptr() + 2, 1, None))
    with pytest.raises(RuntimeError, match="nothing on this stream sets the mark"):
        _lib.check(lib.cg_wait_mark(word.data_ptr(), 1, codec._stream(DEV)))
    with pytest.raises(RuntimeError, match="nothing to move"):
        _lib.check(lib.cg_move_bytes(word.data_ptr(), word.data_ptr(), 0, 1, None, 0, None))


# slots for everything, two and eight in turn; steps of 64 bytes and up; pieces with gaps between them
@pytest.mark.parametrize("slots", [0, 2, 8])
@pytest.mark.parametrize("step,size", [(64, 1000), (4352, 8 * 4352), (4352, 8 * 4352 + 1), (4352, 300001), (2 << 20, (20 << 20) + 77)])
@pytest.mark.parametrize("few", [0, 4 << 20])
def test_staged_pieces_arrive(step, size, slots, few, monkeypatch):
    monkeypatch.setattr(hostmem, "_FEW_BYTES", few)
    print(step, size, slots, flush=True)
    g = torch.Generator().manual_seed(size)
    cuts = sorted({0, size, *(int(x) for x in torch.randint(0, size, (9,), generator=g))})
    if few:
        cuts = cuts[:1] + cuts[-2:]
    pieces = [(a, _bytes(b - a - (1 if b - a > 5 and i % 2 else 0), i)) for i, (a, b) in enumerate(zip(cuts, cuts[1:]))]
    dev = torch.full((size + GUARD,), 8, dtype=torch.uint8, device=DEV)
    with torch.cuda.device(DEV):
        for _ in range(3):
            event = hostmem.event(DEV)
            moves = hostmem.Moves(DEV, codec._stream(DEV))
            moves.stage(pieces, dev.data_ptr(), size, step, slots)
            event.record()
            moves.hold(event)
    got = dev.cpu()
    for at, want in pieces:
        assert torch.equal(got[at:at + want.numel()], want)
    assert (got[size:] == 8).all()


@pytest.mark.parametrize("threads", [0, 1, 3])
def test_staged_pieces_arrive_from_any_team(threads, monkeypatch):
    own = hostmem.team()
    monkeypatch.setattr(hostmem, "team", lambda: hostmem._TEAM.pack(*(hostmem._TEAM.unpack(own)[:2] if threads else (0, 0)), threads, 0))
    monkeypatch.setattr(hostmem, "_FEW_BYTES", 0)
    size = (5 << 20) + 77
    want = _bytes(size, threads)
    dev = torch.zeros(size, dtype=torch.uint8, device=DEV)
    with torch.cuda.device(DEV):
        for slots in (2, 4):
            dev.zero_()
            event = hostmem.event(DEV)
            moves = hostmem.Moves(DEV, codec._stream(DEV))
            moves.stage([(0, want[:1000001]), (1000001, want[1000001:])], dev.data_ptr(), size, 1 << 20, slots)
            event.record()
            moves.hold(event)
            assert torch.equal(dev.cpu(), want)


def test_an_event_is_waited_for_before_it_may_be_recorded_again(monkeypatch):
    """An upload with a stream of its own, whose event the next call gets at once and records behind long work."""
    from cachegen_amd.serde import incoming
    monkeypatch.setattr(incoming, "_WHOLE_BYTES", 1 << 20)
    hold, other, lent = hostmem.Moves.hold, torch.cuda.Stream(), []

    def hold_and_lend(moves, event):
        hold(moves, event)
        event.synchronize()
        with torch.cuda.stream(other):
            torch.cuda._sleep(100_000_000)
            event.record()
        lent.append(event)
    monkeypatch.setattr(hostmem.Moves, "hold", hold_and_lend)
    want = _bytes(3 << 20, 1)
    torch.cuda.synchronize()
    with torch.cuda.device(DEV):
        buf = incoming._upload([(0, want)], (3 << 20) + 64, 3 << 20, lambda base, host: host.zero_())
        arrived = torch.cuda.current_stream().record_event()
    arrived.synchronize()
    assert not lent[0].query(), "the upload was behind another stream's work"
    assert torch.equal(buf[:3 << 20].cpu(), want)


def test_parts_are_filled_as_they_come():
    src = torch.arange(3 << 20, dtype=torch.int32, device=DEV).view(torch.uint8)
    n = src.numel()
    with torch.cuda.device(DEV), hostmem.Moves(DEV, codec._stream(DEV)) as moves:
        a, b = moves.down(src[:n // 3]), moves.down(src[n // 3 + 1:])
        whole = torch.zeros(n, dtype=torch.uint8)
        moves.fill([(whole[:n // 3], *a), (whole[n // 3 + 1:], *b)])
    want = src.cpu()
    want[n // 3] = 0
    assert torch.equal(whole, want)


# tables in one piece and in slices, dense or not, on the GPU or not
@pytest.mark.parametrize("layers,tokens", [(2, 40), (36, 256)])
@pytest.mark.parametrize("form", ["wide", "turned", "host"])
def test_sections_of_any_layout(layers, tokens, form, monkeypatch):
    import dataclasses
    from cachegen_amd.kvgen import make_kv
    from cachegen_amd.serde import wire
    monkeypatch.setattr(wire, "_SLICE_BYTES", 2 << 20)
    bins = torch.full((layers,), 32.0, device=DEV)
    enc = codec.encode_kv(make_kv(layers, tokens, 8, 128, seed=1, device=DEV), bins, bins)
    want = wire.pack_chunks(enc)
    if form == "wide":
        room = torch.zeros((*enc.cdf.shape[:3], enc.cdf.shape[3] + 7), dtype=enc.cdf.dtype, device=DEV)
        other = {"cdf": room[..., :enc.cdf.shape[3]]}
        other["cdf"].copy_(enc.cdf)
    elif form == "turned":
        other = {"cdf": enc.cdf.transpose(1, 2).contiguous().transpose(1, 2), "lengths": enc.lengths.transpose(1, 2).contiguous().transpose(1, 2)}
    else:
        other = {"cdf": enc.cdf.cpu(), "lengths": enc.lengths.cpu(), "maxima": enc.maxima.cpu()}
    assert wire.pack_chunks(dataclasses.replace(enc, **other)) == want


def test_slices_keep_their_place_inside_a_unit(monkeypatch):
    """Tables that begin at no multiple of 16 bytes, in slices: the pinned memory begins at the same place."""
    from cachegen_amd.kvgen import make_kv
    from cachegen_amd.serde import wire
    monkeypatch.setattr(wire, "_SLICE_BYTES", 2 << 20)
    bins = torch.full((1,), 64.0, device=DEV)
    enc = codec.encode_kv(make_kv(1, 16, 20001, 1, seed=1, device=DEV), bins, bins, chunk_tokens=8)
    at = enc.cdf[1].data_ptr()
    assert at % 16 and enc.cdf[1].numel() * 2 > 2 * wire._SLICE_BYTES
    for part in wire.bring_to_host(enc, 1, 1):
        part.arrive()
        assert len(part.slices) > 1 and part.tables.data_ptr() % 16 == at % 16
        assert torch.equal(part.tables.view(torch.int16), enc.cdf[1].cpu().view(-1))


def test_bytes_cross_beside_a_busy_gpu():
    """Moves do not wait for the compute units: 16 MB up and down, in four steps each, while another stream's matrix products
    (0.8 ms each) keep them busy: 0.7 ms, as on a quiet GPU; by launches, each of which waits for the product before it, 6,
    but for one stream in four, which shares the products' hardware queue."""
    a = torch.randn(8192, 8192, dtype=torch.bfloat16, device=DEV)
    c = torch.empty_like(a)
    want, dev = _bytes(16 << 20, 3), torch.empty(16 << 20, dtype=torch.uint8, device=DEV)
    up, down = want.pin_memory(), torch.empty(16 << 20, dtype=torch.uint8, pin_memory=True)
    busy, took = torch.cuda.Stream(), []
    for _ in range(8):
        mine = torch.cuda.Stream()
        torch.cuda.synchronize()
        with torch.cuda.stream(busy):
            for _ in range(30):
                torch.mm(a, a, out=c)
        begin, end = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        with torch.cuda.stream(mine), hostmem.Moves(DEV, codec._stream(DEV)) as moves:
            begin.record()
            for at in range(0, 16 << 20, 4 << 20):
                moves.up(up[at:at + (4 << 20)], dev.data_ptr() + at)
            for at in range(0, 16 << 20, 4 << 20):
                moves.down_to(dev.data_ptr() + at, down[at:at + (4 << 20)])
            end.record()
        end.synchronize()
        took.append(begin.elapsed_time(end))
        assert torch.equal(down, want)
    assert sorted(took)[4] < 2.5, took


def _store_and_retrieve():
    from cachegen_amd.kvgen import make_kv
    from cachegen_amd.serde import incoming, wire
    kv = make_kv(8, 600, 8, 128, seed=1, device=DEV)
    bins = torch.full((8,), 32.0, device=DEV)
    out = torch.empty_like(kv)

    def store():
        return wire.pack_chunks(codec.encode_kv(kv, bins, bins, 256, max_bins=32))

    def retrieve(blobs):
        incoming.decode([(incoming.Container.flat(b), bins, bins, 256 * i) for i, b in enumerate(blobs)], out, "vllm")
        return out
    return store, retrieve


def test_stores_and_retrieves_in_turn_get_no_more_pinned_memory():
    store, retrieve = _store_and_retrieve()
    for i in range(10):
        if i == 3:
            before = torch.cuda.host_memory_stats()["num_host_alloc"]
        retrieve(store())
        torch.cuda.synchronize()
    assert torch.cuda.host_memory_stats()["num_host_alloc"] == before


def test_another_thread_may_capture_meanwhile():
    """Neither new pinned memory nor an event's query gets in the way of a graph that another thread captures."""
    store, retrieve = _store_and_retrieve()
    want, x, got = store(), torch.zeros(1024, device=DEV), []
    for _ in range(3):
        retrieve(store())
    first = retrieve(want).clone()

    def other():
        with torch.cuda.device(DEV):
            got.append(store())
            got.append(retrieve(got[0]).clone())
            torch.cuda.current_stream().synchronize()
    graph = torch.cuda.CUDAGraph()
    torch.cuda.synchronize()
    # (torch.cuda.graph would give the device memory that the calls use back to the system first)
    with torch.cuda.stream(torch.cuda.Stream()):
        graph.capture_begin(capture_error_mode="global")
        x.add_(1)
        t = threading.Thread(target=other)
        t.start()
        t.join()
        x.add_(1)
        graph.capture_end()
    for _ in range(3):
        graph.replay()
    torch.cuda.synchronize()
    assert got[0] == want and torch.equal(got[1], first) and (x == 6).all()
