"""encode_streams_kernel finds a symbol's table entry from the symbol's bits moved to their place in the address: blocks of 64, 128
and 256 lanes, four-bit words of even and odd channels, byte words, rows whose last symbol occurs (saturated,
or a table shorter than the alphabet), sub-chunks that end inside a word and inside a group of eight symbols."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
MANY_WAVEFRONTS, TABLES_IN_CODER = 16, 4


@pytest.mark.parametrize("H,D", [(1, 40), (1, 64), (1, 120), (4, 32), (3, 72), (4, 64), (8, 72)])
@pytest.mark.parametrize("bins,max_bins", [((16.0, 8.0), None), ((32.0, 16.0), None), ((64.0, 16.0), None), ((128.0, 32.0), None),
                                           ((32.0, 16.0), 12), ((16.0, 12.0), 34)])
@pytest.mark.parametrize("saturated", [False, True])
def test_every_place_of_a_symbol(oracle, H, D, bins, max_bins, saturated):
    from cachegen_amd import codec
    T, S = 293, 263                                  # sub-chunks of 256, 7 and 30 tokens
    gen = torch.Generator().manual_seed(H * D)
    kv = torch.rand((2, 2, T, H, D), generator=gen) * 2 - 1
    quiet = torch.rand((1, 1, 1, H, D), generator=gen) < 0.5
    kv = torch.where(quiet, kv * 0.05, kv)
    if saturated:
        kv[0, 0, 31] *= 1e-39                        # MAX / max is infinite: the row's bytes saturate
        kv[1, 1, 260] *= 1e-39
    kv = kv.to(torch.bfloat16)
    kb, vb = torch.tensor(bins), torch.tensor(bins[::-1])
    base = codec.encode_kv(kv.to(DEV), kb, vb, chunk_tokens=S, max_bins=max_bins)
    if max_bins is None and not saturated:           # the reference reads outside its table for a saturated byte: undefined there
        x = kv.view(torch.int16).numpy().view(np.uint16).reshape(2, 2, T, H * D)
        bounds = base.sub_boundaries()
        for ci, c0 in enumerate(range(0, T, S)):
            want = oracle.encode_function(np.ascontiguousarray(x[:, :, c0:c0 + S]), kb.numpy(), vb.numpy(), 1)
            for (b, l, n), (wb, wl, wn) in zip(base.chunk(ci, bounds)[3], want["data_chunks"]):
                assert n == wn and np.array_equal(l.cpu().numpy(), wl) and np.array_equal(b.cpu().numpy(), wb), ci
    for flags in (MANY_WAVEFRONTS, MANY_WAVEFRONTS | TABLES_IN_CODER):
        other = codec.encode_kv(kv.to(DEV), kb, vb, chunk_tokens=S, max_bins=max_bins, _test_flags=flags)
        n = base.total_bytes()
        assert other.total_bytes() == n and int(other.status) == int(base.status)
        assert torch.equal(base.cdf, other.cdf) and torch.equal(base.lengths, other.lengths)
        assert torch.equal(base.payload[:n], other.payload[:n]), flags
