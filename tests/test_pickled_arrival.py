"""The pickle writer takes a tensor's bytes only once they have arrived: small tensors, which stand in
the pickle itself, large ones, which are copied into the blob, and a mixture."""
import pytest
import torch

from cachegen_amd.serde.cachegen_basics import CacheGenGPUBytestream, CacheGenGPUEncoderOutput
from cachegen_amd.serde import pickled


@pytest.mark.parametrize("rows, C, tokens", [(4, 16, 40), (4, 8192, 40), (8, 4096, 4200)])
def test_bytes_are_read_after_arrival(rows, C, tokens):
    L, lp = rows // 2, 33
    make = torch.Generator().manual_seed(rows * C + tokens)
    shapes = [((777777 if C > 1000 else 99,), torch.uint8), ((rows, C), torch.int32), ((rows, C, lp), torch.int16),
              ((L, tokens, 1), torch.float16), ((L, tokens, 1), torch.float16)]
    want = [torch.randint(0, 256, (n * t.itemsize,), generator=make, dtype=torch.uint8)
            for n, t in ((torch.Size(s).numel(), t) for s, t in shapes)]
    host = [w.clone() if i >= 3 else torch.zeros_like(w) for i, w in enumerate(want)]     # the maxima are there
    calls = []

    def arrive():
        calls.append(1)
        for h, w in zip(host, want):
            h.copy_(w)

    w = pickled._Writer("cpu", arrive)
    stream, lengths, cdf, key, value = (w.tensor(h, t, s, there=i >= 3) for i, (h, (s, t)) in enumerate(zip(host, shapes)))
    blob = w.finish(CacheGenGPUEncoderOutput([CacheGenGPUBytestream(stream, lengths, tokens)], cdf, max_tensors_key=key,
                                             max_tensors_value=value, num_heads=1, head_size=C))
    out = CacheGenGPUEncoderOutput.from_bytes(blob)
    got = [out.data_chunks[0].bytestream, out.data_chunks[0].bytestream_lengths, out.cdf, out.max_tensors_key, out.max_tensors_value]
    assert calls
    for g, b, (s, t) in zip(got, want, shapes):
        assert tuple(g.shape) == s and g.dtype is t
        assert torch.equal(g.contiguous().view(torch.uint8).reshape(-1), b)
