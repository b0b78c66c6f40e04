"""Streams made to lead the float32 search astray (decoder.hpp: decode_symbol<..., FLOAT>): a symbol followed by 24 bits
or more of the lowest symbol leaves the code value within a few parts in 2^24 of the symbol's lower bound, where
the search may fall short by one entry, and one followed by the highest symbol leaves it as close below the upper bound,
where it may overshoot.  On the CPU: such streams do both, at the last entry of a half table, at the
last symbol and next to it.  On the GPU: they decode to what was encoded."""
import numpy as np
import pytest
import torch

from cachegen_amd import codec
from test_fast_forms_model import Reader, corrected, float_search
from test_kernel_arithmetic_model import M32, step_count

DEV = "cuda:0"
TOKENS, CHANNELS, ROWS = 251, 1024, 6
# what the row's levels say -> (levels, highest symbol that is coded, search steps left out, the last symbol may occur)
KINDS = {"half": lambda lp: ((lp - 1) // 2, (lp - 1) // 2 - 1, 1, False),
         "next to the last": lambda lp: (lp - 1, lp - 3, 0, False),
         "last": lambda lp: (2 * (lp - 1), lp - 2, 0, True)}


def streams(oracle, lp, kind, channels=CHANNELS):
    """(tables uint16 [ROWS, channels, lp], symbols uint8 [ROWS, TOKENS, channels]): every few symbols one of the highest
    ones, a random one or 1, the rest the lowest symbol, in odd channels the highest."""
    _, top, _, _ = KINDS[kind](lp)
    rng = np.random.default_rng(lp)
    bits = lp.bit_length() - 1
    cdf = oracle.calculate_cdf(rng.integers(0, lp - 1, size=(ROWS, 2048, channels), dtype=np.uint8), lp - 1)   # even tables
    sym = np.zeros((ROWS, TOKENS, channels), dtype=np.uint8)
    sym[:, :, 1::2] = top
    every = -(-26 // bits) + 1
    for first in range(every):                                 # the cycle begins anywhere
        at = np.arange(first, TOKENS, every)
        some = rng.integers(1, top + 1, size=(ROWS, len(at), channels))
        sure = rng.choice([top, max(1, top - 1), 1], size=some.shape)
        sym[:, at, first::every] = np.where(rng.random(some.shape) < 0.5, some, sure)[:, :, first::every]
    return cdf, sym


def guesses(cdf, log2, skip, safe, data, n):
    """(symbol, guess of the float search) of every symbol that is not coded in the full range."""
    rd, low, span, out, off = Reader(data, 0), 0, 0, [], None
    off = rd.off
    for _ in range(n):
        rd.top_up()
        if span == 0:
            m = max(k for k in range(len(cdf) - 1) if cdf[k] << 16 <= off)
            t_lo, width = cdf[m] << 16, ((0x10000 if m == len(cdf) - 2 else cdf[m + 1]) - cdf[m]) << 16
            low, guess = 0, m
        else:
            guess = float_search(cdf, log2, skip, span, off)
            m, t_lo, width, _ = corrected(cdf, log2, skip, safe, span, off, guess)
        out.append((m, guess))
        low, off, d = (low + t_lo) & M32, off - t_lo, (width - 1) & M32
        k = step_count(low, (low + d) & M32, d)
        low, span = (low << k) & M32, (width << k) & M32
        off = ((off << 32 | rd.win >> 32) << k) >> 32 & M32
        rd.win = rd.win << k & (1 << 64) - 1
        rd.bits -= k
    return out


@pytest.mark.parametrize("lp", [9, 17, 33, 65])
@pytest.mark.parametrize("kind", list(KINDS))
def test_streams_lead_the_search_astray(oracle, lp, kind):
    _, top, skip, safe = KINDS[kind](lp)
    cdf, sym = streams(oracle, lp, kind, channels=8)
    padded, lengths = oracle.encode_fast_new(cdf, sym)
    short, over = [], []
    for r in range(ROWS):
        for c in range(8):
            data = padded[r, c, :lengths[r, c]].tobytes()
            got = guesses([int(x) for x in cdf[r, c]], lp.bit_length() - 1, skip, safe, data, TOKENS)
            assert [m for m, _ in got] == list(sym[r, :, c])
            short += [m for m, guess in got if guess == m - 1]
            over += [m for m, guess in got if guess == m + 1]
    assert short.count(top) >= 5                               # the search's last entry, the last symbol, the one next to it
    if safe:
        assert len(over) >= 5 and max(over) == top - 1         # from the symbol below the last


@pytest.mark.gpu
@pytest.mark.parametrize("lp", [9, 17, 33, 65])
@pytest.mark.parametrize("kind", list(KINDS))
def test_streams_come_back(oracle, lp, kind):
    levels, _, _, _ = KINDS[kind](lp)
    cdf, sym = streams(oracle, lp, kind)
    padded, lengths = oracle.encode_fast_new(cdf, sym)
    assert lengths.max() <= 256
    units = torch.cuda.get_device_properties(0).multi_processor_count
    # four wavefronts a SIMD: more than decode_few_kernel takes, fewer than decode_streams_kernel
    reps = units * 4 * 4 // (ROWS * CHANNELS // 64)
    L, layers_of = reps * ROWS // 2, torch.arange(reps * ROWS, device=DEV) % ROWS
    kept = np.arange(256)[None, None, :] < lengths[..., None]
    payload = torch.from_numpy(padded[..., :256][kept]).to(DEV).repeat(reps)
    lengths = torch.from_numpy(lengths.astype(np.int64)).to(DEV)[layers_of]
    offsets = torch.cat([lengths.new_zeros(1), lengths.flatten().cumsum(0)])
    tables = torch.from_numpy(cdf.view(np.int16)).to(DEV)[layers_of][None]
    gen = torch.Generator(DEV).manual_seed(lp)
    maxima = (torch.rand(2, L, TOKENS, device=DEV, generator=gen) + 0.5).half()
    bins = torch.full((L,), float(levels), device=DEV)
    got = codec.decode_kv(tables, maxima, offsets, payload, bins, bins, L, TOKENS, CHANNELS // 128, 128, TOKENS, out_dtype=torch.float16)
    # (s - C) / C * maximum in float32, rounded once more (decoder.py:28-34); rows are keys of all layers, then values
    c = levels // 2 - 1
    quotients = (torch.arange(256, device=DEV, dtype=torch.float32) - c) / c
    symbols = torch.from_numpy(sym).to(DEV).long()[layers_of].view(2, L, TOKENS, CHANNELS)
    want = (quotients[symbols] * maxima.float()[..., None]).half().permute(1, 0, 2, 3).reshape(got.shape)
    assert torch.equal(got.view(torch.int16), want.contiguous().view(torch.int16))
