"""Containers decoded together by one launch (cg_decode_listed, serde/incoming.py) against the
whole-tensor decoder on each of them: channel counts around a wavefront and a block, token counts
around a sub-chunk, table lengths and containers mixed in one call, uploads in one piece and in many."""
import numpy as np
import pytest
import torch

from cachegen_amd import codec
from cachegen_amd.kvgen import make_kv
from cachegen_amd.serde import incoming, wire

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("H,D", [(1, 8), (1, 64), (5, 24), (3, 43), (9, 64)])       # 8, 64, 120, 129 (odd), 576 channels
@pytest.mark.parametrize("fmt", ["vllm", "huggingface"])
def test_containers_of_several_kinds_in_one_call(H, D, fmt, monkeypatch):
    L = 3
    if H * D > 500:
        monkeypatch.setattr(incoming, "_WHOLE_BYTES", 1 << 16)
        monkeypatch.setattr(incoming, "_PIECE_BYTES", 4352)                  # pieces that cut sections anywhere
    cases = [(1, 256, (32, 16, 16), "flat"), (256, 256, (16, 12, 8), "compact"), (257, 300, (32, 32, 32), "compact"),
             (600, 256, (64, 32, 32), "flat"), (77, 77, (32, 16, 16), "compact"), (513, 128, (8, 8, 8), "compact")]
    tdim = 2 if fmt == "vllm" else 3
    items, wants, t0 = [], [], 0
    for k, (T, S, bins, kind) in enumerate(cases):
        kv = make_kv(L, T, H, D, seed=k, device=DEV, dtype=torch.bfloat16 if k % 2 else torch.float16)
        kb, vb = torch.tensor([float(b) for b in bins]), torch.tensor([float(b) for b in bins[::-1]])
        enc = codec.encode_kv(kv, kb, vb, chunk_tokens=S)
        blob = wire.pack_chunks(enc, per_chunk=False, compact=kind == "compact")[0]
        if k % 3 == 0:
            kb, vb = kb.to(DEV), vb.to(DEV)                                  # levels on the device and on the host
        items.append((incoming.Container.flat(blob), kb, vb, t0))
        wants.append(codec.decode_encoded(enc, kb, vb, fmt=fmt, out_dtype=torch.bfloat16))
        t0 += T
    shape = list(wants[0].shape)
    shape[tdim] = t0
    out = torch.full(shape, float("nan"), dtype=torch.bfloat16, device=DEV)
    incoming.decode(items, out, fmt)
    want = torch.cat(wants, dim=tdim)
    assert torch.equal(out.view(torch.int16), want.view(torch.int16))


@pytest.mark.parametrize("dtype", ["<i4", "<u2"])
@pytest.mark.parametrize("C", [1, 63, 64, 65, 200])
def test_running_sums_on_the_host(dtype, C):
    from cachegen_amd import _lib
    nsub, rows, tiles = 3, 4, -(-C // 64)
    lengths = np.random.default_rng(C).integers(0, 400, size=(nsub, rows, C)).astype(dtype)
    starts, total = np.empty((nsub, rows, tiles), dtype=np.uint32), np.empty(nsub, dtype=np.int64)
    args = (lengths.ctypes.data, lengths.itemsize, nsub, rows, C, starts.ctypes.data, total.ctypes.data)
    assert _lib.lib().cg_host_tile_starts(*args) == 0
    stored = np.minimum(lengths, 256).astype(np.int64).reshape(nsub, -1)
    before = (np.cumsum(stored, axis=1) - stored).reshape(nsub, rows, C)[:, :, ::64]
    assert np.array_equal(starts, before) and np.array_equal(total, stored.sum(axis=1))
    if dtype == "<i4":
        lengths[2, 3, C - 1] = -1
        assert _lib.lib().cg_host_tile_starts(*args) != 0
