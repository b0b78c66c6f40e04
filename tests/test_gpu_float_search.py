"""Decodes on both sides of the line between decode_float_kernel and decode_streams_kernel (twelve
wavefronts a SIMD, tables of 64 symbols never the latter): the same streams decoded in one large call
and in calls of a few to twelve wavefronts a SIMD give the same bits."""
import pytest
import torch

from cachegen_amd import codec

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def wavefronts(per_simd):
    return torch.cuda.get_device_properties(0).multi_processor_count * 4 * per_simd


@pytest.mark.parametrize("bins", [(8.0, 6.0), (16.0, 9.0), (32.0, 16.0), (64.0, 33.0), (16.0, 16.0)])
@pytest.mark.parametrize("H,D", [(8, 128), (5, 80), (1, 40)])          # whole blocks, ragged ones, blocks of one wavefront
@pytest.mark.parametrize("fmt", ["vllm", "huggingface"])
def test_large_and_smaller_decodes_agree(bins, H, D, fmt):
    L = 24 if H > 1 else 120
    per_sub = 2 * L * -(-H * D // 64)
    nsub = wavefronts(12) // per_sub + 1                       # the least sub-chunks of the large side
    T = (nsub - 1) * 256 + 77
    gen = torch.Generator(DEV).manual_seed(4)
    spread = torch.rand(L, 2, 1, H, D, device=DEV, generator=gen) ** 4 + 0.01     # quiet channels and loud ones
    kv = torch.empty(L, 2, T, H, D, device=DEV, dtype=torch.bfloat16).normal_(generator=gen).mul_(spread.bfloat16())
    kv[0, 0, 300] *= 2.0 ** -126                               # saturates: the table's last symbol, in one sub-chunk
    kv[1, 1, 600, 0, 0] = float("inf")
    if fmt == "huggingface":
        kv = kv.permute(0, 1, 3, 2, 4).contiguous()
    dim = 2 if fmt == "vllm" else 3
    kb = torch.tensor([bins[i % 2] for i in range(L)], device=DEV)
    vb = torch.tensor([bins[1 - i % 2] for i in range(L)], device=DEV)
    top = int(bins[0])
    enc = codec.encode_kv(kv, kb, vb, chunk_tokens=256, fmt=fmt, max_bins=top)
    whole = codec.decode_encoded(enc, kb, vb, fmt=fmt, out_dtype=torch.float16)
    per_call = wavefronts(4) // per_sub + 1                    # more than the few-wavefront form takes
    for a, n in ((0, per_call), (1, per_call + 3), (nsub - per_call, per_call), (0, nsub - 1)):
        part = kv.narrow(dim, a * 256, min(n * 256, T - a * 256)).contiguous()
        got = codec.decode_encoded(codec.encode_kv(part, kb, vb, chunk_tokens=256, fmt=fmt, max_bins=top), kb, vb, fmt=fmt, out_dtype=torch.float16)
        want = whole.narrow(dim, a * 256, part.shape[dim])
        nan = torch.isnan(want)
        assert torch.equal(torch.isnan(got), nan)
        assert torch.equal(got.view(torch.int16)[~nan], want.contiguous().view(torch.int16)[~nan])


@pytest.mark.parametrize("top", [8, 16, 32, 64])
@pytest.mark.parametrize("delta_group", [0, 10])
def test_streams_of_rare_symbols_come_back(top, delta_group):
    """Uniform values: every step of the search, and more bits a symbol than the window is made for."""
    L, T, H, D = 2, 3 * 256 + 9, 8, 128
    reps = wavefronts(4) // (2 * L * 16 * 4) + 1
    gen = torch.Generator(DEV).manual_seed(top)
    kv = (torch.rand(L, 2, T, H, D, device=DEV, generator=gen) * 2 - 1).half()
    bins = torch.full((L,), float(top), device=DEV)
    small = codec.decode_encoded(codec.encode_kv(kv, bins, bins, chunk_tokens=T, max_bins=top, delta_group=delta_group), bins, bins,
                                 fmt="vllm", out_dtype=torch.float16)
    many = kv.repeat(reps, 1, 1, 1, 1)
    bins = torch.full((L * reps,), float(top), device=DEV)
    enc = codec.encode_kv(many, bins, bins, chunk_tokens=T, max_bins=top, delta_group=delta_group)
    got = codec.decode_encoded(enc, bins, bins, fmt="vllm", out_dtype=torch.float16)
    step = 2.0 / (2 * (top // 2 - 1))                          # of the quantizer; a delta adds its anchor's error
    assert float((got[:L].float() - kv.float()).abs().max()) < step * (1.01 if delta_group == 0 else 2.6)
    for r in range(reps):
        assert torch.equal(got[r * L:(r + 1) * L].view(torch.int16), small.view(torch.int16))
