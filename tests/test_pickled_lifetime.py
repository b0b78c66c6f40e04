"""Reading a pickle container lets go of the blob: nothing of it stays behind once the container is dropped."""
import gc
import pickle
import struct
import sys

import pytest
import torch

from cachegen_amd.serde import pickled
from cachegen_amd.serde.cachegen_basics import CacheGenGPUBytestream, CacheGenGPUEncoderOutput


@pytest.mark.parametrize("plain", [True, False])        # False: refused (one chunk too few), left to the plain unpickler
def test_a_blob_is_free_after_it_was_read(plain):
    L, C, T, lp = 2, 64, 300, 33
    chunks = [CacheGenGPUBytestream(torch.zeros(n, dtype=torch.uint8), torch.zeros((2 * L, C), dtype=torch.int32), t)
              for n, t in ((100000, 256), (1000, T - 256))]
    maxima = [torch.zeros((L, T, 1), dtype=torch.float16) for _ in range(2)]
    blob = CacheGenGPUEncoderOutput(chunks if plain else chunks[:1], torch.zeros((2 * L, C, lp), dtype=torch.int16),
                                    max_tensors_key=maxima[0], max_tensors_value=maxima[1], num_heads=1, head_size=C).to_bytes()
    gc.collect()
    before = sys.getrefcount(blob)
    for _ in range(3):
        container = pickled.container(blob)
        assert (container is not None) == plain
        del container
    assert sys.getrefcount(blob) == before


@pytest.mark.parametrize("module,name", [("torch._utils", "_rebuild_tensor_v2"), ("torch.storage", "_load_from_bytes")])
@pytest.mark.parametrize("state", [{"mark": 1}, (None, {"__defaults__": (1,)}), (None, {"__kwdefaults__": {"mark": 1}})])
def test_a_blob_changes_nothing_that_outlives_it(module, name, state):
    """BUILD sets attributes of the object below it on the stack, here of what stands in for torch's function."""
    given = pickled._tensor, pickled._storage
    before = [(dict(f.__dict__), f.__defaults__, f.__kwdefaults__) for f in given]
    body = ("c%s\n%s\n" % (module, name)).encode() + pickle.dumps(state, protocol=2)[2:-1] + b"b."
    blob = b"\x80\x04\x95" + struct.pack("<Q", len(body)) + body
    assert pickled.container(blob) is None
    assert [(dict(f.__dict__), f.__defaults__, f.__kwdefaults__) for f in given] == before
