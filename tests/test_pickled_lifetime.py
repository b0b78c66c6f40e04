"""Reading a pickle container lets go of the blob: nothing of it stays behind once the container is dropped."""
import gc
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
