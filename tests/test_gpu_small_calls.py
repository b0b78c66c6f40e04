"""The forms that calls of few blocks take: tables counted by slices of a block, payload places added
up from all tile counts, streams of a padded buffer packed by one launch."""
import numpy as np
import pytest
import torch

from cachegen_amd import codec, torchac_hip
from cachegen_amd.kvgen import make_kv

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("nl,nc,cap", [(1, 1, 8), (2, 5, 64), (3, 127, 256), (4, 512, 100)])
def test_streams_of_a_padded_buffer_are_packed(nl, nc, cap):
    rng = np.random.default_rng(nc)
    padded = rng.integers(0, 256, size=(nl, nc, cap + 3), dtype=np.uint8)[:, :, :cap]
    lengths = rng.integers(0, cap + 1, size=(nl, nc)).astype(np.int32)
    lengths[0, 0] = cap
    device = torch.from_numpy(np.ascontiguousarray(padded)).to(DEV)
    wide = torch.zeros((nl, nc + 1, cap + 3), dtype=torch.uint8, device=DEV)
    wide[:, :nc, :cap] = device
    want = np.concatenate([padded[r, c, :lengths[r, c]] for r in range(nl) for c in range(nc)])
    offsets = codec.scan_lengths(torch.from_numpy(lengths).to(DEV))
    for buffer in (device, wide[:, :nc, :cap]):
        assert np.array_equal(codec.collect_streams(buffer, offsets).cpu().numpy(), want)
    assert codec.collect_streams(device, torch.zeros_like(offsets)).numel() == 0


@pytest.mark.parametrize("nt", [1, 7, 8, 9, 31, 32, 33, 255, 256, 1000])
@pytest.mark.parametrize("nc", [40, 300])
def test_tables_counted_by_slices(oracle, nt, nc):
    sym = np.random.default_rng(nt).integers(0, 20, size=(2, nt, nc)).astype(np.uint8)
    got = torchac_hip.calculate_cdf(torch.from_numpy(sym.view(np.int8)).to(DEV), 32)
    assert np.array_equal(got.cpu().numpy().view(np.uint16), oracle.calculate_cdf(sym, 32))


@pytest.mark.parametrize("nsub", [1, 2, 511, 512, 513])      # two tiles each: around the 1024 tiles added up directly
@pytest.mark.parametrize("chunk", [256, 512])
def test_payload_places_from_all_tile_counts(nsub, chunk):
    kv = make_kv(1, nsub * 256 - 3, 2, 128, seed=nsub, device=DEV) if nsub < 100 else \
        torch.randn(1, 2, nsub * 256 - 3, 2, 128, device=DEV, generator=torch.Generator(DEV).manual_seed(nsub)).half()
    bins = torch.tensor([16.0], device=DEV)
    a = codec.encode_kv(kv, bins, bins, chunk_tokens=chunk, _test_flags=4)          # tables in the coder or a pass of their own
    b = codec.encode_kv(kv, bins, bins, chunk_tokens=chunk, _test_flags=2)          # tables in the quantizer
    a.check()
    n = a.total_bytes()
    assert n == b.total_bytes() == int(a.lengths.sum())
    assert torch.equal(a.offsets, b.offsets) and torch.equal(a.payload[:n], b.payload[:n]) and torch.equal(a.cdf, b.cdf)
