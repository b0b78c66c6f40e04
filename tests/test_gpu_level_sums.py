"""Payload places from group sums that the packing quantizer clears, on both sides of the 1024 tiles up to
which all tile counts are added up: every level equals a separate encode, and one whose tables the
quantizer makes."""
import pytest
import torch

from cachegen_amd import codec

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("nsub", [127, 128, 129, 140])                  # eight tiles each
@pytest.mark.parametrize("nlevels", [1, 3, 8])
def test_levels_and_separate_encodes_agree(nsub, nlevels):
    L, T, H, D = 4, nsub * 256 - 5, 2, 128
    kv = torch.randn(L, 2, T, H, D, device=DEV, generator=torch.Generator(DEV).manual_seed(nsub)).half()
    tops = [(8, 16, 32, 64)[v % 4] for v in range(nlevels)]
    levels = [(torch.full((L,), float(t), device=DEV), torch.full((L,), float(t // 2), device=DEV)) for t in tops]
    for _ in range(2):                                                  # sums left by the call before
        encs = codec.encode_kv_levels(kv, levels, chunk_tokens=256, max_bins=tops)
    for (kb, vb), top, e in zip(levels, tops, encs):
        e.check()
        n = e.total_bytes()
        for flags in (4, 2):                                            # tables in the coder, in the quantizer
            one = codec.encode_kv(kv, kb, vb, chunk_tokens=256, max_bins=top, _test_flags=flags)
            assert torch.equal(e.offsets, one.offsets) and torch.equal(e.payload[:n], one.payload[:n]) and torch.equal(e.cdf, one.cdf)
