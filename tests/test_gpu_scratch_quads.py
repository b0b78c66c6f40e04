"""The encoder's scratch holds streams in quads of four words, or word by word where sub-chunks have at most 48 tokens, and the
compaction takes eight words at a time: streams that end on either side of a quad, ranges of several LDS tiles, long
streams among short ones, in launches of few and of many blocks."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
MANY_WAVEFRONTS = 16


@pytest.mark.parametrize("L,T,H,D,S,bins", [
    (2, 4112, 4, 64, 16, (64.0, 16.0)),         # 1028 tiles (the few-block form takes 1024) of streams of 2 to 14 bytes
    (2, 4097, 4, 64, 33, (64.0, 32.0)),         # 500 tiles, the last chunk has five tokens
    (1, 300, 4, 64, 300, (64.0,)),              # two tiles, streams of up to 200 bytes
    (1, 512, 3, 40, 64, (64.0,)),               # 120 channels: tiles that straddle rows
    (1, 21, 5, 40, 7, (128.0,)),                # tables of 129 entries, blocks of 128 lanes
    (2, 197, 4, 64, 48, (64.0, 32.0)),          # word by word: the longest sub-chunks, of streams past eight words
    (2, 197, 4, 64, 49, (64.0, 32.0)),          # the shortest in quads
    (1, 144, 5, 40, 48, (64.0,)),               # tiles that straddle rows: both again
    (1, 147, 5, 40, 49, (64.0,)),
    (2, 48, 4, 64, 1500, (64.0, 16.0)),         # one chunk, short by its tokens
    (1, 48, 1, 64, 48, (128.0,)),               # idle lanes, a tile of several rows
])
def test_streams_of_any_length_beside_one_another(oracle, L, T, H, D, S, bins):
    from cachegen_amd import codec
    gen = torch.Generator().manual_seed(T)
    kv = torch.rand((L, 2, T, H, D), generator=gen) * 2 - 1               # the whole alphabet alike: the longest streams
    quiet = torch.rand((1, 1, 1, H, D), generator=gen) < 0.7
    kv = torch.where(quiet, kv * 0.02, kv)                                # the centre symbol only, nearly
    kv = kv.to(torch.float16)
    kb, vb = torch.tensor((bins * L)[:L]), torch.tensor((bins[::-1] * L)[:L])
    x = kv.view(torch.int16).numpy().view(np.uint16).reshape(L, 2, T, H * D)
    for flags in (0, MANY_WAVEFRONTS):
        enc = codec.encode_kv(kv.to(DEV), kb, vb, chunk_tokens=S, _test_flags=flags)
        enc.check()
        bounds = enc.sub_boundaries()
        for ci, c0 in enumerate(range(0, T, S)):
            want = oracle.encode_function(np.ascontiguousarray(x[:, :, c0:c0 + S]), kb.numpy(), vb.numpy(), 0)
            _, _, _, subs = enc.chunk(ci, bounds)
            for (b, l, n), (wb, wl, wn) in zip(subs, want["data_chunks"]):
                assert n == wn and np.array_equal(l.cpu().numpy(), wl) and np.array_equal(b.cpu().numpy(), wb), (flags, ci)
