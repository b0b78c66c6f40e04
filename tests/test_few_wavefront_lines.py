"""Up to how many blocks an encode takes the coder's form for few wavefronts (encode_few_kernel): no more than
a compute unit's LDS holds at once, for every table length, and the same streams on both sides of
each line."""
import pytest
import torch

from cachegen_amd import _lib, codec, torchac_hip
from cachegen_amd.kvgen import make_kv

BYTES, COUNTED, TABLES, QUANTIZER_TABLES = range(4)
DEV = "cuda:0"


def blocks(source, lp, block, tile=False):
    return _lib.lib().cg_test_few_encode_blocks(source, lp, block, tile)


@pytest.mark.parametrize("source", range(4))
@pytest.mark.parametrize("block,tile", [(64, False), (128, False), (256, False), (256, True)])
def test_blocks_fit_a_compute_unit(source, block, tile):
    for lp in range(2, 130):
        n = blocks(source, lp, block, tile)
        lds = lp * block * 4 + (0 if source == BYTES else 272)       # 32-bit entries, one column a lane
        assert n >= 0 and n * (-(-lds // 1280) * 1280) <= 160 * 1024
        assert n * block <= (12 if source == BYTES else 8) * 64      # the registers for a sub-chunk's symbols
        assert lp == 2 or n <= blocks(source, lp - 1, block, tile)


def test_lines_of_the_measured_lengths():
    assert [blocks(BYTES, lp, 256) for lp in (17, 33, 34, 65, 79)] == [3, 3, 2, 2, 2]
    assert [blocks(BYTES, lp, 128) for lp in (81, 97, 113, 129)] == [3, 3, 2, 2]
    assert [blocks(COUNTED, lp, 256, True) for lp in (17, 33, 65, 80)] == [2, 2, 2, 1]
    assert [blocks(COUNTED, lp, 256) for lp in (17, 33, 65)] == [2, 2, 1]
    assert [blocks(COUNTED, lp, 128) for lp in (17, 65, 81, 129)] == [2, 2, 1, 1]
    assert [blocks(COUNTED, lp, 64) for lp in (17, 65)] == [2, 2]
    assert [blocks(TABLES, lp, 256, True) for lp in (17, 33, 65, 80)] == [2, 1, 1, 1]
    assert [blocks(TABLES, lp, 256) for lp in (17, 29, 33)] == [2, 1, 0]
    assert [blocks(QUANTIZER_TABLES, lp, 256, True) for lp in (17, 33, 65)] == [2, 2, 1]
    assert [blocks(QUANTIZER_TABLES, lp, 256) for lp in (17, 33, 65)] == [2, 1, 0]
    for source in (TABLES, QUANTIZER_TABLES):
        assert [blocks(source, lp, 128) for lp in (17, 33, 81)] == [2, 0, 0] and blocks(source, 17, 64) == 0
    for args in ((-1, 33, 256), (4, 33, 256), (BYTES, 1, 256), (BYTES, 130, 256), (BYTES, 33, 32)):
        assert blocks(*args) == -1


def units():
    return torch.cuda.get_device_properties(0).multi_processor_count


@pytest.mark.gpu
@pytest.mark.parametrize("lp", [17, 33, 34, 52, 53, 65, 80, 81, 106, 128])
def test_byte_symbols_on_both_sides(lp):
    C, T, block = 256, 77, 256 if lp <= 80 else 128
    most = units() * blocks(BYTES, lp, block) * block // C           # rows that take the form for few wavefronts
    gen = torch.Generator(DEV).manual_seed(lp)
    sym = (torch.randn(most + 1, T, C, device=DEV, generator=gen) * lp / 8 + lp / 2).clamp(0, lp - 2).to(torch.uint8)
    cdf = torchac_hip.calculate_cdf(sym, lp - 1)
    got = []
    for rows in (most, most + 1):
        out = torch.zeros((rows, C, 256), dtype=torch.uint8, device=DEV)
        lengths = torch.zeros((rows, C), dtype=torch.int32, device=DEV)
        torchac_hip.encode_fast_new(cdf[:rows], sym[:rows], out, lengths)
        got.append((out, lengths))
    assert torch.equal(got[0][0], got[1][0][:most]) and torch.equal(got[0][1], got[1][1][:most])
    back = torch.full_like(sym, 255)
    torchac_hip.decode_fast_new(cdf, got[1][0], got[1][1], back)
    assert torch.equal(back, sym)


@pytest.mark.gpu
@pytest.mark.parametrize("source,T,S,flags,top", [(COUNTED, 90, 256, 0, t) for t in (16, 32, 64, 79, 96, 128)] +
                         [(TABLES, 300, 300, 4, t) for t in (16, 32, 64, 79, 96, 128)] +
                         [(QUANTIZER_TABLES, 90, 256, 2, t) for t in (16, 32, 64)])
@pytest.mark.parametrize("H,D", [(4, 64), (5, 80), (1, 128), (1, 64)])       # a whole tile, blocks of 256, 128 and 64 lanes
def test_packed_symbols_on_both_sides(source, T, S, flags, top, H, D):
    C = H * D
    block = 64 if C == 64 else 128 if C == 128 or top >= 80 else 256
    per_layer = 2 * -(-C // block) * -(-T // 256)
    most = units() * blocks(source, top + 1, block, block == 256 and C == 256) // per_layer      # layers
    for L in (max(1, most), most + 1):
        kv = make_kv(L, T, H, D, seed=top, device=DEV, dtype=torch.bfloat16)
        bins = torch.full((L,), float(top), device=DEV)
        a = codec.encode_kv(kv, bins, bins, chunk_tokens=S, max_bins=top, _test_flags=flags)
        b = codec.encode_kv(kv, bins, bins, chunk_tokens=S, max_bins=top, _test_flags=flags | 16)   # CG_TEST_MANY_WAVEFRONTS
        a.check()
        n = a.total_bytes()
        assert n == b.total_bytes() and torch.equal(a.payload[:n], b.payload[:n])
        assert torch.equal(a.cdf, b.cdf) and torch.equal(a.lengths, b.lengths) and torch.equal(a.offsets, b.offsets)
