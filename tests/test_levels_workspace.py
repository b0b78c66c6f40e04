"""What several levels ask of memory: the larger and the least workspace, and which calls can use the larger one."""
import ctypes

import pytest

from cachegen_amd import _lib, codec

SYMBOLS = 256                        # bytes a stream of 256 tokens; its scratch as many


@pytest.mark.parametrize("L,T,C,S,n", [(32, 4096, 1024, 256, 4), (1, 1, 8, 16, 8), (32, 16384, 1024, 256, 4), (80, 32768, 1024, 256, 4), (32, 16640, 1024, 256, 2)])
def test_workspaces(L, T, C, S, n):
    least, wanted = codec.encode_levels_least_workspace_bytes(L, T, C, S, n), codec.encode_levels_workspace_bytes(L, T, C, S, n)
    streams = codec.num_subchunks(T, S) * 2 * L * C
    tiles = -(-streams // 256)
    one = codec.encode_workspace_bytes(L, T, C, S)
    # symbols for every level and what one level needs beside its symbols: an encode of one level, and symbols for the others
    assert abs(least - (one + (n - 1) * streams * SYMBOLS)) <= n * 1024 + 256 * n
    extra = (n - 1) * (one - streams * SYMBOLS)
    assert abs(wanted - least - (extra if tiles <= 16384 else 0)) <= n * 1024 + 256 * n
    assert codec.encode_levels_least_workspace_bytes(L, T, C, S, 1) == codec.encode_levels_workspace_bytes(L, T, C, S, 1)


@pytest.mark.parametrize("H,D,L,T,tops,together", [
    (8, 128, 32, 4096, (8, 64), True),
    (8, 128, 32, 4096, (8,), False),             # one level
    (8, 128, 32, 4096, (8, 80), False),          # a table of 81 entries: blocks of 128 lanes
    (1, 128, 32, 4096, (8, 64), False),          # few channels: the same
    (8, 100, 32, 4096, (8, 64), False),          # no vector loads
    (8, 128, 80, 32768, (8, 64), False),         # above the line of the larger workspace
])
def test_which_calls_share_launches(H, D, L, T, tops, together):
    got = _lib.lib().cg_encode_kv_levels_together(4096, L, T, H, D, 2 * T * H * D, T * H * D, H * D, D, len(tops),
                                                  (ctypes.c_int * len(tops))(*tops), 256)
    assert bool(got) is together
