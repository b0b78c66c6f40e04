"""Encodes on both sides of the line between encode_few_kernel and encode_streams_kernel: the same
tables, lengths and bytes, against the oracle where the four-at-a-time path gives way to the exact one
(more bits than it holds, the full range again and again, the last symbol); such streams decoded
on both sides too."""
import numpy as np
import pytest
import torch

from cachegen_amd import codec, torchac_hip
from cachegen_amd.kvgen import make_kv

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
MANY = 16                                                     # CG_TEST_MANY_WAVEFRONTS


def same(a, b):
    a.check()
    n = a.total_bytes()
    return (n == b.total_bytes() and torch.equal(a.cdf, b.cdf) and torch.equal(a.lengths, b.lengths) and
            torch.equal(a.offsets, b.offsets) and torch.equal(a.payload[:n], b.payload[:n]))


# channels that are whole tiles of 256 and that are not, tables made by the coder and by a pass of their own
@pytest.mark.parametrize("H,D", [(4, 64), (5, 80), (1, 40)])
@pytest.mark.parametrize("T,S", [(1, 256), (7, 256), (8, 256), (127, 256), (129, 256), (135, 256), (136, 256), (255, 256), (700, 256), (300, 300), (513, 600)])
@pytest.mark.parametrize("bins", [(32.0, 16.0), (64.0, 33.0), (16.0, 8.0)])
def test_both_forms_give_the_same_streams(H, D, T, S, bins):
    for dtype in (torch.float16, torch.bfloat16):
        kv = make_kv(2, T, H, D, seed=T + D, device=DEV, dtype=dtype)
        kv[0, :, 0] *= 1e-30 if dtype == torch.bfloat16 else 0          # a row that saturates (or is zero)
        if dtype == torch.bfloat16:
            kv[1, 1, T // 2] *= 2.0 ** -126
        kb, vb = torch.tensor([bins[0], bins[1]], device=DEV), torch.tensor([bins[1], bins[0]], device=DEV)
        for flags in (0, 1, 4):
            few = codec.encode_kv(kv, kb, vb, chunk_tokens=S, max_bins=int(bins[0]), _test_flags=flags)
            many = codec.encode_kv(kv, kb, vb, chunk_tokens=S, max_bins=int(bins[0]), _test_flags=flags | MANY)
            assert same(few, many)


def encoded(cdf, sym, cap):
    lengths = torch.zeros((sym.shape[0], sym.shape[2]), dtype=torch.int32, device=DEV)
    out = torch.full((sym.shape[0], sym.shape[2], cap), 0xEE, dtype=torch.uint8, device=DEV)
    torchac_hip.encode_fast_new(cdf, sym, out, lengths)
    return lengths.cpu().numpy(), out.cpu().numpy()


@pytest.mark.parametrize("nt", [0, 1, 3, 4, 5, 8, 12, 63, 64, 65, 77, 128, 200, 256])
@pytest.mark.parametrize("kind", ["rare", "dyadic", "mixed"])
@pytest.mark.parametrize("cap", [256, 640])
def test_streams_of_many_bits_match_oracle(oracle, nt, kind, cap):
    rng = np.random.default_rng(nt)
    nl, nc = 2, 70
    if kind == "dyadic":                                      # every interval scales back to the full range
        cdf = np.broadcast_to(np.append(np.arange(16) * 4096, 65535).astype(np.uint16), (nl, nc, 17)).copy()
        sym = rng.integers(0, 16, size=(nl, nt, nc)).astype(np.uint8)
    else:                                                     # tables made of one symbol: the others take 16 bits each
        seen = np.full((nl, 256, nc), 3, dtype=np.uint8)
        if kind == "mixed":
            seen[:, ::2] = rng.integers(0, 16, size=seen[:, ::2].shape)
        cdf = oracle.calculate_cdf(seen, 16)
        sym = rng.integers(0, 16, size=(nl, nt, nc)).astype(np.uint8)
        sym[:, :, ::3] = 3                                    # beside streams of next to no bits
    want_pad, want_len = oracle.encode_fast_new(cdf, sym, cap=cap)
    d_cdf, d_sym = torch.from_numpy(cdf.view(np.int16)).to(DEV), torch.from_numpy(sym.view(np.int8)).to(DEV)
    kept = np.arange(cap)[None, None, :] < np.minimum(want_len, cap)[..., None]
    rows = torch.cuda.get_device_properties(0).multi_processor_count * 4 * 3      # more wavefronts than the few
    for reps in (1, rows // nl):
        lengths, out = encoded(d_cdf.repeat(reps, 1, 1), d_sym.repeat(reps, 1, 1), cap)
        for r in {0, reps // 2, reps - 1}:
            got_len, got = lengths[r * nl:(r + 1) * nl], out[r * nl:(r + 1) * nl]
            assert np.array_equal(got_len, want_len)
            assert np.array_equal(got[kept], want_pad[kept]) and (got[~kept] == 0xEE).all()
        if cap == 640 and nt:                                 # whole streams: and back, also four at a time and one by one
            back = torch.full((reps * nl, nt, nc), 255, dtype=torch.uint8, device=DEV)
            torchac_hip.decode_fast_new(d_cdf.repeat(reps, 1, 1), torch.from_numpy(out).to(DEV), torch.from_numpy(lengths).to(DEV), back)
            assert torch.equal(back.view(torch.int8), d_sym.repeat(reps, 1, 1))
