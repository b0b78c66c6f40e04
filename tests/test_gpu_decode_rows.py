"""decode_streams_kernel's unrolled search begins with a choice between two addresses that it holds in registers (tables of 9, 17
and 33 entries; rows that use the lower half of their table, and rows that use all of it), in calls of more wavefronts than the
forms for few take: blocks of 64 and 128 lanes, with idle lanes, symbols and dequantised values, a row whose last
symbol occurs (bfloat16: a scale that overflows).  Tables of 65 entries (decode_float_kernel) and of other lengths (the search
without those probes) go the same way through the same calls beside them."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("H,D,nsub,S", [(8, 128, 200, 7), (1, 40, 3100, 5), (3, 72, 800, 9)])      # over 12 wavefronts a SIMD each
@pytest.mark.parametrize("bins", [(8.0, 8.0), (16.0, 12.0), (32.0, 16.0), (64.0, 32.0), (24.0, 16.0)])
@pytest.mark.parametrize("dtype,dt", [(torch.float16, 0), (torch.bfloat16, 1)])
def test_dequantised_values(oracle, H, D, nsub, S, bins, dtype, dt):
    from cachegen_amd import codec
    L, T = 2, nsub * S - 1                                   # the last chunk is one token short
    gen = torch.Generator().manual_seed(H * D + S)
    kv = torch.rand((L, 2, T, H, D), generator=gen) * 2 - 1
    kv = kv.to(dtype)
    if dtype is torch.bfloat16:
        kv[1, 1, 3 * S] *= 1e-39                             # the scale overflows at any level: the table's last symbol
    kb, vb = torch.tensor(bins), torch.tensor(bins[::-1])
    max_bins = int(max(bins))
    dev = kv.to(DEV)
    enc = codec.encode_kv(dev, kb, vb, chunk_tokens=S)
    out = codec.decode_encoded(enc, kb, vb, fmt="vllm", out_dtype=dtype)
    sym, maxima = codec.quantize_kv(dev, kb.to(DEV), vb.to(DEV))
    saturated = sym[L + 1, 3 * S] == 255
    assert bool(saturated.any()) == (dtype is torch.bfloat16)
    sym = np.minimum(sym.cpu().numpy(), max_bins - 1)        # bytes outside the table are its last symbol
    mx = maxima.cpu().view(torch.int16).numpy().view(np.uint16)
    got = out.cpu().view(torch.int16).numpy().view(np.uint16).reshape(L, 2, T, H * D)
    assert np.array_equal(got[:, 0], oracle.dequantize(sym[:L], kb.numpy(), mx[0], dt, dt))
    assert np.array_equal(got[:, 1], oracle.dequantize(sym[L:], vb.numpy(), mx[1], dt, dt))


@pytest.mark.parametrize("rows,channels,tokens", [(210, 1024, 9), (3300, 40, 6), (1700, 120, 11)])      # over 3 wavefronts a SIMD each
@pytest.mark.parametrize("max_bins", [8, 16, 32, 64, 23, 100])
def test_symbols(rows, channels, tokens, max_bins):
    from cachegen_amd import torchac_hip
    from cachegen_amd.serde.cachegen_basics import CacheGenGPUBytestream
    from cachegen_amd.serde.cachegen_decoder import decode_chunk
    from cachegen_amd.serde.cachegen_encoder import encode_ntokens
    gen = torch.Generator().manual_seed(rows)
    sym = torch.randint(0, max_bins, (rows, tokens, channels), generator=gen).to(torch.int8).to(DEV)
    cdf = torchac_hip.calculate_cdf(sym, max_bins)
    buffer = torch.zeros((rows, channels, 256), dtype=torch.uint8, device=DEV)
    lengths = torch.zeros((rows, channels), dtype=torch.int32, device=DEV)
    stream = encode_ntokens(cdf, sym, buffer, lengths)
    out = torch.zeros((rows, tokens, channels), dtype=torch.uint8, device=DEV)
    decode_chunk(cdf, CacheGenGPUBytestream(stream, lengths, tokens), out)
    assert torch.equal(out, sym.view(torch.uint8))
