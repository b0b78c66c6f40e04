"""Decodes on both sides of the line between decode_few_kernel (calls of at most three wavefronts a SIMD)
and decode_streams_kernel: the same streams decoded in one large call and in small ones give the
same bits, for every table length that has both, whole and ragged sub-chunks."""
import pytest
import torch

from cachegen_amd import codec, torchac_hip
from cachegen_amd.kvgen import make_kv
from cachegen_amd.serde.cachegen_basics import CacheGenGPUBytestream
from cachegen_amd.serde.cachegen_decoder import decode_chunk
from cachegen_amd.serde.cachegen_encoder import encode_ntokens

pytestmark = pytest.mark.gpu


def most_wavefronts():
    return torch.cuda.get_device_properties(0).multi_processor_count * 4 * 3


@pytest.mark.parametrize("bins", [(16.0, 9.0), (32.0, 16.0), (64.0, 33.0)])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_one_large_decode_equals_small_ones(bins, dtype):
    dev, L, H, D = "cuda:0", 3, 8, 128
    per_sub = 2 * L * (H * D // 64)
    nsub = most_wavefronts() // per_sub + 1                    # the least sub-chunks of the large side
    T = (nsub - 1) * 256 + 77
    kv = make_kv(L, T, H, D, seed=9, device=dev, dtype=dtype)
    kb = torch.tensor([bins[0], bins[1], bins[0]], device=dev)
    vb = torch.tensor([bins[1], bins[0], bins[1]], device=dev)
    top = int(bins[0])
    whole = codec.decode_encoded(codec.encode_kv(kv, kb, vb, chunk_tokens=256, max_bins=top), kb, vb, fmt="vllm", out_dtype=dtype)
    step = (nsub - 1) * 256                                    # as many wavefronts as the small side takes
    for a, b in ((0, step), (step, T), (256, 256 + 3), (512, 512 + 13 * 256 + 130)):
        part = kv[:, :, a:b].contiguous()
        got = codec.decode_encoded(codec.encode_kv(part, kb, vb, chunk_tokens=256, max_bins=top), kb, vb, fmt="vllm", out_dtype=dtype)
        if b - a == 3 or (b - a) % 256 and b != T:             # tables of its own for the last, cut chunk
            b = a + (b - a) // 256 * 256
        assert torch.equal(got[:, :, :b - a].view(torch.int16), whole[:, :, a:b].view(torch.int16))


@pytest.mark.parametrize("top", [16, 32, 64])
@pytest.mark.parametrize("tokens", [1, 7, 8, 129, 256])
def test_symbols_come_back_on_both_sides(top, tokens):
    dev, C = "cuda:0", 200                                     # four wavefronts a row, the last one with 8 lanes
    edge = most_wavefronts() // 4
    gen = torch.Generator().manual_seed(tokens)
    for rows in (5, edge, edge + 1):
        # symbols around the middle, the whole alphabet (the last symbol included) in a few channels
        sym = (torch.randn(rows, tokens, C, generator=gen) * 1.5 + top // 2).clamp(0, top - 1)
        sym[:, :, ::37] = torch.randint(0, top, sym[:, :, ::37].shape, generator=gen).float()
        sym = sym.to(torch.int8).to(dev)
        cdf = torchac_hip.calculate_cdf(sym, top)
        buffer = torch.zeros((rows, C, 256), dtype=torch.uint8, device=dev)
        lengths = torch.zeros((rows, C), dtype=torch.int32, device=dev)
        stream = encode_ntokens(cdf, sym, buffer, lengths)
        out = torch.full((rows, tokens, C), 255, dtype=torch.uint8, device=dev)
        decode_chunk(cdf, CacheGenGPUBytestream(stream, lengths, tokens), out)
        assert torch.equal(out.view(torch.int8), sym)
