"""Levels of one cache coded by shared launches (cg_encode_kv_levels): every way the levels are dealt to
launches gives the bytes of a separate encode at each level."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _bins(top, L):
    """Two tiers: `top` bins in the first third of the layers, half of that in the others."""
    b = torch.full((L,), max(4.0, top / 2))
    b[:(L + 2) // 3] = top
    return b


# (layers, tokens, heads, head size), chunk, largest bins of each level
CASES = [
    ((1, 1, 1, 8), 16, (8, 16)),                  # one stream tile, mostly empty
    ((2, 33, 8, 64), 16, (64, 8, 32)),            # few wavefronts, three chunks, the last one token
    ((3, 257, 5, 80), 256, (16, 32, 64)),         # channels that fill no tile: offsets from a scan
    ((4, 520, 8, 128), 260, (8, 16, 32, 64)),     # tables of two sub-chunks, all levels resident at once
    ((6, 2048, 8, 128), 256, (8, 64, 32, 60)),    # more blocks than are resident: launches by table length
    ((6, 2048, 8, 128), 40, (8, 64, 32)),         # the same with scratch laid word by word
    ((6, 2048, 8, 128), 700, (64, 8)),            # the same with tables made by a pass of their own
    ((2, 300, 8, 128), 256, (16, 96)),            # a table too long for blocks of 256 lanes: one launch each
    ((4, 256, 8, 128), 256, (8, 16, 24, 32, 40, 48, 56, 64)),
]


@pytest.mark.parametrize("shape,chunk,tops", CASES)
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_levels_in_shared_launches(shape, chunk, tops, dtype):
    from cachegen_amd import codec
    from cachegen_amd.kvgen import make_kv
    L, T, H, D = shape
    kv = make_kv(L, T, H, D, seed=5 + T, device=DEV, dtype=dtype)
    levels = [(_bins(float(t), L), _bins(float(t), L)) for t in tops]
    print(dict(shape=shape, chunk=chunk, tops=tops, dtype=str(dtype)), flush=True)
    got = codec.encode_kv_levels(kv, levels, chunk_tokens=chunk)
    for (kb, vb), e in zip(levels, got):
        want = codec.encode_kv(kv, kb, vb, chunk_tokens=chunk)
        n = want.total_bytes()
        assert e.total_bytes() == n and int(e.status) == int(want.status) == 0
        for name in ("cdf", "maxima", "lengths", "offsets"):
            assert torch.equal(getattr(e, name), getattr(want, name)), name
        assert torch.equal(e.payload[:n], want.payload[:n])


def _levels_and_cache(seed):
    from cachegen_amd.kvgen import make_kv
    kv = make_kv(6, 2048, 8, 128, seed=seed, device=DEV, dtype=torch.float16)      # two launches, one beside the other
    return kv, [(_bins(float(t), 6).to(DEV), _bins(float(t), 6).to(DEV)) for t in (8, 64, 32)]


def _bytes(encs):
    return [t.clone() for e in encs for t in (e.cdf, e.lengths, e.offsets, e.payload[:e.total_bytes()])]


def test_levels_in_a_graph():
    from cachegen_amd import codec
    kv, levels = _levels_and_cache(1)
    tops = [8, 64, 32]
    ws = torch.empty(codec.encode_levels_workspace_bytes(6, 2048, 1024, 256, 3), dtype=torch.uint8, device=DEV)
    out = codec.encode_kv_levels(kv, levels, chunk_tokens=256, max_bins=tops, workspace=ws)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        codec.encode_kv_levels(kv, levels, chunk_tokens=256, max_bins=tops, workspace=ws, out=out)
    for seed in (2, 3, 4):
        other, _ = _levels_and_cache(seed)
        want = _bytes(codec.encode_kv_levels(other, levels, chunk_tokens=256, max_bins=tops))
        kv.copy_(other)
        graph.replay()
        assert all(torch.equal(a, b) for a, b in zip(_bytes(out), want))


def test_levels_on_several_streams_at_once():
    """More callers than there are side streams; each call's inputs are written just before it and dropped just behind."""
    import threading
    from cachegen_amd import codec
    tops = [8, 64, 32]
    want = {seed: _bytes(codec.encode_kv_levels(*_levels_and_cache(seed), chunk_tokens=256, max_bins=tops)) for seed in (1, 2, 3)}
    torch.cuda.synchronize()
    wrong = []

    def caller(seed):
        with torch.cuda.stream(torch.cuda.Stream()):
            for _ in range(6):
                kv, levels = _levels_and_cache(seed)
                got = codec.encode_kv_levels(kv, levels, chunk_tokens=256, max_bins=tops)
                del kv, levels
                if not all(torch.equal(a, b) for a, b in zip(_bytes(got), want[seed])):
                    wrong.append(seed)
    callers = [threading.Thread(target=caller, args=(seed,)) for seed in want]
    for c in callers:
        c.start()
    for c in callers:
        c.join()
    assert not wrong


def test_a_call_does_not_wait_for_another_streams_work():
    from cachegen_amd import codec
    tops = [8, 64, 32]
    kv, levels = _levels_and_cache(1)
    want = _bytes(codec.encode_kv_levels(kv, levels, chunk_tokens=256, max_bins=tops))
    first, second = torch.cuda.Stream(), torch.cuda.Stream()
    torch.cuda.synchronize()
    with torch.cuda.stream(first):
        torch.cuda._sleep(100_000_000)
        late = codec.encode_kv_levels(kv, levels, chunk_tokens=256, max_bins=tops)
        last = first.record_event()
    with torch.cuda.stream(second):
        got = codec.encode_kv_levels(kv, levels, chunk_tokens=256, max_bins=tops)
        through = second.record_event()
    through.synchronize()
    assert not last.query(), "the second call was behind the first stream's work"
    torch.cuda.synchronize()
    for encs in (late, got):
        assert all(torch.equal(a, b) for a, b in zip(_bytes(encs), want))


@pytest.mark.parametrize("shape,chunk,tops", [c for c in CASES if len(c[2]) > 1])
def test_levels_with_the_least_workspace(shape, chunk, tops):
    """Levels that share one scratch, one behind the other; nothing behind the workspace is written."""
    from cachegen_amd import codec
    from cachegen_amd.kvgen import make_kv
    L, T, H, D = shape
    kv = make_kv(L, T, H, D, seed=3 + T, device=DEV, dtype=torch.float16)
    levels = [(_bins(float(t), L), _bins(float(t), L)) for t in tops]
    n = codec.encode_levels_least_workspace_bytes(L, T, H * D, chunk, len(tops))
    assert n < codec.encode_levels_workspace_bytes(L, T, H * D, chunk, len(tops))
    room = torch.full((n + 4096,), 7, dtype=torch.uint8, device=DEV)
    print(dict(shape=shape, chunk=chunk, tops=tops), flush=True)
    want = _bytes(codec.encode_kv_levels(kv, levels, chunk_tokens=chunk))
    got = codec.encode_kv_levels(kv, levels, chunk_tokens=chunk, workspace=room[:n])
    assert all(torch.equal(a, b) for a, b in zip(_bytes(got), want))
    assert (room[n:] == 7).all()


def test_a_gpu_without_room_for_the_larger_workspace(monkeypatch):
    from cachegen_amd import codec
    kv, levels = _levels_and_cache(1)
    want = _bytes(codec.encode_kv_levels(kv, levels, chunk_tokens=256))
    large = codec.encode_levels_workspace_bytes(6, 2048, 1024, 256, 3)
    empty, asked = torch.empty, []

    def little(*size, **kw):
        if size == (large,):
            asked.append(size)
            raise torch.cuda.OutOfMemoryError
        return empty(*size, **kw)
    monkeypatch.setattr(torch, "empty", little)
    got = codec.encode_kv_levels(kv, levels, chunk_tokens=256)
    assert asked and all(torch.equal(a, b) for a, b in zip(_bytes(got), want))
