"""Tables <-> histogram counts on the GPU against the numpy forms: channel counts around a block of 64,
table lengths from the smallest to the largest, token counts at which the divisions can go wrong, more
groups than a grid has rows."""
import numpy as np
import pytest
import torch

from cachegen_amd import _lib
from cachegen_amd.serde import wire

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("C", [1, 63, 64, 65, 200])
@pytest.mark.parametrize("lp", [2, 3, 33, 129])
def test_counts_and_tables(C, lp):
    lib, stream = _lib.lib(), torch.cuda.current_stream().cuda_stream
    rng = np.random.default_rng(C * lp)
    tokens = [1, 2, 3, 255, 256]
    rows, G = 2, 10
    counts = np.zeros((len(tokens), rows, C, lp - 1), dtype=np.int64)
    for k, n in enumerate(tokens):
        for r in range(rows):
            top = rng.integers(1, lp)                                        # symbols that occur, fewer in some groups
            for c in range(C):
                counts[k, r, c] = np.bincount(rng.integers(0, top, n) if c % 3 else np.full(n, top - 1), minlength=lp - 1)
    cdf = wire.counts_to_tables(counts, tokens)
    tables = torch.from_numpy(cdf.view(np.int16)).to(DEV)
    tok = torch.from_numpy(np.repeat(np.asarray(tokens, dtype=np.int32), rows)).to(DEV)
    dense = torch.empty((G, C, lp - 1), dtype=torch.uint8, device=DEV)
    nsym = torch.empty(G, dtype=torch.int32, device=DEV)
    inexact = torch.empty(1, dtype=torch.int32, device=DEV)
    _lib.check(lib.cg_tables_to_counts(tables.data_ptr(), lp - 1, G, C, tok.data_ptr(), dense.data_ptr(), nsym.data_ptr(),
                                       inexact.data_ptr(), stream))
    want = np.minimum(counts, 255).astype(np.uint8).reshape(G, C, lp - 1)
    symbols = np.array([1 + max(np.flatnonzero(want[g].any(axis=0))) for g in range(G)])
    assert inexact.item() == 0 and np.array_equal(dense.cpu().numpy(), want) and np.array_equal(nsym.cpu().numpy(), symbols)
    ragged = np.concatenate([want[g, :, :symbols[g]].ravel() for g in range(G)])
    packed = torch.empty(ragged.size, dtype=torch.uint8, device=DEV)
    _lib.check(lib.cg_pack_counts(dense.data_ptr(), lp - 1, G, C, nsym.data_ptr(), None, packed.data_ptr(), stream))
    assert np.array_equal(packed.cpu().numpy(), ragged)
    starts = torch.from_numpy(np.cumsum(symbols * C) - symbols * C).to(DEV)
    stored = nsym.to(torch.uint8)
    back, invalid = torch.empty_like(tables), torch.empty(1, dtype=torch.int32, device=DEV)
    for wrong in (0, 1):
        if wrong:
            packed[-1] ^= 64                                                 # the last channel no longer adds up
        _lib.check(lib.cg_counts_to_tables(packed.data_ptr(), ragged.size, lp - 1, G, C, tok.data_ptr(), stored.data_ptr(),
                                           starts.data_ptr(), back.data_ptr(), invalid.data_ptr(), stream))
        assert invalid.item() == wrong
        assert wrong or torch.equal(back, tables)
    tables.view(-1)[lp - 1] ^= 1                                             # not what any histogram gives
    _lib.check(lib.cg_tables_to_counts(tables.data_ptr(), lp - 1, G, C, tok.data_ptr(), dense.data_ptr(), nsym.data_ptr(),
                                       inexact.data_ptr(), stream))
    assert inexact.item() == 1


def test_more_groups_than_a_grid_has_rows():
    lib, stream = _lib.lib(), torch.cuda.current_stream().cuda_stream
    G = 65537
    tokens = np.arange(G, dtype=np.int32) % 255 + 1
    data, tok = torch.from_numpy(tokens.astype(np.uint8)).to(DEV), torch.from_numpy(tokens).to(DEV)
    one, starts = torch.ones(G, dtype=torch.uint8, device=DEV), torch.arange(G, dtype=torch.int64, device=DEV)
    cdf, invalid = torch.empty((G, 1, 3), dtype=torch.int16, device=DEV), torch.empty(1, dtype=torch.int32, device=DEV)
    _lib.check(lib.cg_counts_to_tables(data.data_ptr(), G, 2, G, 1, tok.data_ptr(), one.data_ptr(), starts.data_ptr(),
                                       cdf.data_ptr(), invalid.data_ptr(), stream))
    assert invalid.item() == 0
    assert (cdf.view(-1, 3) == torch.tensor([0, -2, -1], dtype=torch.int16, device=DEV)).all()
