"""Words that kernels store for a host that looks at their mark: numbers read back, the largest bins, the sizes of a
collect_bytes and the decode from lengths, at the edges of their launches."""
import math
import threading

import pytest
import torch

from cachegen_amd import codec, hostmem, torchac_hip
from cachegen_amd.serde.cachegen_encoder import collect_bytes

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("dtype", [torch.int32, torch.int64])
def test_numbers_are_read_back(dtype):
    t = torch.tensor([-1, 2 ** 31 - 1, -2 ** 31, 7, 0], dtype=dtype, device=DEV)
    assert [hostmem.read_number(t, i) for i in range(-5, 5)] == 2 * t.tolist()
    assert [hostmem.read_number(t[::2], i) for i in range(3)] == t[::2].tolist()
    with pytest.raises(IndexError):
        hostmem.read_number(t, 5)
    for k in range(50):                                     # behind work that is still queued
        t.fill_(k)
        assert hostmem.read_number(t, 3) == k


def test_each_thread_reads_its_own():
    wrong = []

    def reader(i):
        stream = torch.cuda.Stream()
        with torch.cuda.stream(stream):
            t = torch.empty(3, dtype=torch.int64, device=DEV)
            for k in range(200):
                t.fill_(1000 * i + k)
                if hostmem.read_number(t, 1) != 1000 * i + k:
                    wrong.append((i, k))
    threads = [threading.Thread(target=reader, args=(i,)) for i in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not wrong


@pytest.mark.parametrize("n", [1, 2, 63, 64, 65, 200])
def test_largest_of_two_vectors(n):
    g = torch.Generator().manual_seed(n)
    for place in (0, n // 2, n - 1):
        a, b = torch.rand(n, generator=g) * 30 - 40, torch.rand(n, generator=g) * 30 - 40
        (a if place % 2 else b)[place] = 33.75
        assert codec._largest(a.to(DEV), b.to(DEV)) == 33
        assert codec._largest(-a.to(DEV).abs() - 1, -b.to(DEV).abs() - 1) == int(max((-a.abs() - 1).max(), (-b.abs() - 1).max()))
        a[place] = math.nan
        with pytest.raises(ValueError):
            codec._largest(a.to(DEV), b.to(DEV))
    with pytest.raises(OverflowError):
        codec._largest(torch.full((n,), math.inf, device=DEV), b.to(DEV))


# one length, a thread's sixteen, a block's 16384 and one more (several launches), slots to spare and too few
@pytest.mark.parametrize("rows,cols", [(1, 1), (3, 5), (1, 1025), (2, 8192), (1, 16385)])
def test_streams_are_collected(rows, cols):
    cap = 32
    g = torch.Generator().manual_seed(rows * cols)
    padded = torch.randint(0, 256, (rows, cols, cap), generator=g, dtype=torch.uint8)
    lengths = torch.randint(0, cap + 1, (rows, cols), generator=g, dtype=torch.int32)
    lengths[-1, -1] = cap
    keep = torch.arange(cap) < lengths[..., None]
    got = collect_bytes(padded.to(DEV), lengths.to(DEV))
    assert torch.equal(got.cpu(), padded[keep])
    few = lengths.view(-1)[:max(1, rows * cols - 3)].to(DEV)
    assert torch.equal(collect_bytes(padded.to(DEV), few).cpu(), padded.view(-1, cap)[:few.numel()][keep.view(-1, cap)[:few.numel()]])
    bad = lengths.clone()
    bad.view(-1)[rows * cols // 2] = cap + 1
    with pytest.raises(RuntimeError, match="do not fit"):
        collect_bytes(padded.to(DEV), bad.to(DEV))
    with pytest.raises(RuntimeError, match="do not fit"):
        collect_bytes(padded.to(DEV), torch.cat([lengths.view(-1), torch.ones(1, dtype=torch.int32)]).to(DEV))
    assert collect_bytes(padded.to(DEV), torch.zeros_like(lengths).to(DEV)).numel() == 0


@pytest.mark.parametrize("rows,cols,tokens", [(1, 64, 1), (4, 100, 33), (2, 1500, 256), (20, 1024, 16)])
def test_decode_from_lengths(rows, cols, tokens):
    sym = torch.randint(0, 31, (rows, tokens, cols), generator=torch.Generator().manual_seed(cols), dtype=torch.int8).to(DEV)
    cdf = torchac_hip.calculate_cdf(sym, 32)
    buf = torch.zeros((rows, cols, 256), dtype=torch.uint8, device=DEV)
    lengths = torch.zeros((rows, cols), dtype=torch.int32, device=DEV)
    torchac_hip.encode_fast_new(cdf, sym, buf, lengths)
    stream = collect_bytes(buf, lengths)
    out = torch.zeros(sym.shape, dtype=torch.uint8, device=DEV)
    torchac_hip.decode_fast_lengths(cdf, stream, lengths, out)
    assert torch.equal(out, sym.view(torch.uint8))


def test_words_are_used_again_after_an_error():
    hostmem.read_number(torch.zeros(1, dtype=torch.int32, device=DEV), 0)
    kept, lost = len(hostmem._free.words), len(hostmem.Words._lost)
    with pytest.raises(KeyError):
        with hostmem.Words() as words:
            words.set(codec._stream(torch.device(DEV))).synchronize()
            raise KeyError
    assert (len(hostmem._free.words), len(hostmem.Words._lost)) == (kept, lost)
    with pytest.raises(KeyError):
        with hostmem.Words():
            raise KeyError                              # nothing was launched, which nobody can know
    assert (len(hostmem._free.words), len(hostmem.Words._lost)) == (kept - 1, lost + 1)


def test_a_pickle_of_small_tensors():
    from cachegen_amd.kvgen import make_kv
    from cachegen_amd.serde import pickled
    from cachegen_amd.serde.cachegen_basics import CacheGenGPUEncoderOutput
    bins = torch.full((1,), 8.0)
    enc = codec.encode_kv(make_kv(1, 9, 1, 8, seed=1, device=DEV), bins, bins)
    out = CacheGenGPUEncoderOutput.from_bytes(pickled.pack_chunks(enc)[0])
    assert torch.equal(out.cdf.to(DEV), enc.cdf[0]) and torch.equal(out.data_chunks[0].bytestream.to(DEV), enc.payload[:enc.total_bytes()])
