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


@pytest.mark.parametrize("dtype", [torch.uint8, torch.int8, torch.int32])
@pytest.mark.parametrize("shape", [(40,), (5, 40), (3, 4, 40), (2, 3, 2, 40)])
def test_padded_buffers_of_any_rank_and_type_are_packed(dtype, shape):
    """As gathering the streams one by one does it, also with fewer lengths than slots and with empty
    streams behind the last slot."""
    from cachegen_amd.serde.cachegen_encoder import collect_bytes
    rng = np.random.default_rng(len(shape))
    padded = rng.integers(-100, 100, size=shape).astype(np.int32)
    slots = padded.reshape(-1, 40)
    device = torch.from_numpy(padded).to(dtype).to(DEV)
    for n in {1, len(slots) - 1 or 1, len(slots), len(slots) + 3}:
        lengths = rng.integers(0, 41, size=n).astype(np.int32)
        lengths[len(slots):] = 0
        want = torch.from_numpy(np.concatenate([slots[g, :lengths[g]] for g in range(min(n, len(slots)))])).to(dtype)
        got = collect_bytes(device, torch.from_numpy(lengths).to(DEV))
        assert got.dtype == dtype and torch.equal(got.cpu(), want)


@pytest.mark.parametrize("lengths", [[8, 9, 8, 8], [8, 8, 8, 300], [0, 0, 0, 0, 1], [8, 8, 8, 8, 0, 2]])
def test_lengths_that_do_not_fit_the_padded_buffer_are_refused(lengths):
    from cachegen_amd.serde.cachegen_encoder import collect_bytes
    padded = torch.zeros((2, 2, 8), dtype=torch.uint8, device=DEV)
    with pytest.raises(RuntimeError, match="do not fit 4 slots of 8"):
        collect_bytes(padded, torch.tensor(lengths, dtype=torch.int32, device=DEV))
    with pytest.raises(RuntimeError, match="do not fit 4 slots of 8"):
        codec.collect_streams(padded, torch.tensor([1, 2, 3, 4, 5], device=DEV))         # does not begin at 0


# both sides of the lines of sliced_lanes (launch.hpp): rows of 1024 channels, tokens of a chunk
@pytest.mark.parametrize("nt,rows", [(63, 64), (63, 65), (64, 128), (64, 129), (511, 128), (511, 129), (512, 256), (512, 257)])
def test_tables_of_bytes_on_both_sides_of_the_slices_line(oracle, nt, rows):
    sym = np.random.default_rng(nt).integers(0, 20, size=(rows, nt, 1024), dtype=np.uint8)
    got = torchac_hip.calculate_cdf(torch.from_numpy(sym.view(np.int8)).to(DEV), 32)
    assert np.array_equal(got.cpu().numpy().view(np.uint16), oracle.calculate_cdf(sym, 32))


@pytest.mark.parametrize("chunk,tokens", [(639, 1278), (639, 1279), (640, 2560), (640, 2561), (5000, 4097)])
def test_packed_tables_on_both_sides_of_the_slices_line(chunk, tokens):
    """16 layers of 1024 channels: two and four chunks are the lines' 64 k and 128 k lanes."""
    kv = torch.randn(16, 2, tokens, 8, 128, device=DEV, generator=torch.Generator(DEV).manual_seed(tokens)).half()
    bins = torch.full((16,), 32.0, device=DEV)
    a, b = (codec.encode_kv(kv, bins, bins, chunk_tokens=chunk, _test_flags=f) for f in (4, 2))      # a pass of their own, the quantizer
    n = a.total_bytes()
    assert torch.equal(a.cdf, b.cdf) and n == b.total_bytes() and torch.equal(a.payload[:n], b.payload[:n])
