"""What the containers' readers and writers do with the calls they were not tuned for: outputs they
cannot write, levels of any type and stride, levels that a program changes, and errors between a launch
and the host's look at what it stored."""
import types

import pytest
import torch

from cachegen_amd import hostmem
from cachegen_amd.serde import incoming

DEV = "cuda:0"


@pytest.fixture
def order(monkeypatch):
    """Stands in for the stream and for pinned memory where there is no GPU; lists what happens."""
    seen = []
    event = types.SimpleNamespace(synchronize=lambda: seen.append("event waited for"))
    stream = types.SimpleNamespace(synchronize=lambda: seen.append("stream waited for"), record_event=lambda: event)
    zeros = torch.zeros
    monkeypatch.setattr(torch.cuda, "current_stream", lambda: stream)
    monkeypatch.setattr(torch, "zeros", lambda *a, pin_memory=False, **kw: zeros(*a, **kw))
    return seen


@pytest.mark.parametrize("launched", [False, True])
def test_words_that_kernels_store_to_are_held_until_the_launches_are_through(order, launched):
    with pytest.raises(KeyError):
        with hostmem.StoredWords(2, torch.int64) as words:
            if launched:
                words.stored()
            raise KeyError
    assert order == ["event waited for" if launched else "stream waited for"]
    with hostmem.StoredWords(2, torch.int64) as words:
        words.stored()
        assert words.read() == [0, 0]


@pytest.mark.parametrize("out,tokens", [(torch.zeros(2, 2, 300, 2, 8), 0), (torch.zeros(2, 2, 300, 2, 9).half(), 0),
                                        (torch.zeros(3, 2, 300, 2, 8).half(), 0), (torch.zeros(2, 2, 299, 2, 8).half(), 0),
                                        (torch.zeros(2, 2, 300, 2, 8).half(), 1), (torch.zeros(2, 2, 300, 2, 8).half(), -1),
                                        (torch.zeros(2, 2, 300, 2, 16).half()[..., ::2], 0)])
def test_outputs_that_cannot_be_written_are_refused_before_anything_is_queued(out, tokens, monkeypatch):
    monkeypatch.setattr(incoming, "_upload", lambda *a: pytest.fail("something was queued"))
    container = incoming.Container(2, 300, 2, 8, 256, 32, 0, False, False)
    container.payload_bytes = 1
    bins = torch.full((2,), 32.0)
    with pytest.raises(RuntimeError, match="output tensor does not match|must be contiguous"):
        incoming.decode([(container, bins, bins, tokens)], out, "vllm")


@pytest.mark.gpu
def test_counts_that_make_no_table_are_refused_and_leave_the_reader_usable():
    from cachegen_amd.kvgen import make_kv
    from cachegen_amd.config import LMCacheEngineConfig, LMCacheEngineMetadata
    from cachegen_amd.serde import CreateSerde, wire
    s, d = CreateSerde("cachegen-compact", LMCacheEngineConfig.from_defaults(chunk_size=256),
                       LMCacheEngineMetadata("lmsys/longchat-7b-16k", 1, 0, "vllm"))
    blob = s.to_bytes(make_kv(32, 256, 2, 64, seed=3, device=DEV))
    want = d.from_bytes(blob)
    at = wire.read_header(blob)["geometry"]["cdf"][0] + 64 + 7          # a count: 64 rows' symbol counts come first
    bad = bytearray(blob)
    bad[at] = (bad[at] + 1) % 200
    with pytest.raises(ValueError, match="add up"):
        d.from_bytes(bytes(bad))
    assert torch.equal(d.from_bytes(blob), want)
    with pytest.raises(RuntimeError, match="output tensor does not match"):
        d.from_bytes_into(blob, torch.empty(want.shape, device=DEV))
    assert torch.equal(d.from_bytes(blob), want)


@pytest.mark.parametrize("offsets,match", [(torch.zeros(5, dtype=torch.int32), "offsets must be"), (torch.zeros((5, 1), dtype=torch.int64), "offsets must be"),
                                           (torch.zeros(10, dtype=torch.int64)[::2], "offsets must be"), (torch.zeros(1, dtype=torch.int64), "offsets must be"),
                                           (torch.zeros(5, dtype=torch.int64), "on the same GPU")])
def test_offsets_that_the_packing_kernel_would_misread_are_refused(offsets, match):
    from cachegen_amd import codec
    with pytest.raises(RuntimeError, match=match):
        codec.collect_streams(torch.zeros((2, 2, 8), dtype=torch.uint8), offsets)
    with pytest.raises(RuntimeError, match="lengths should be int32"):
        codec.scan_lengths(offsets)


FORMS = {"strided": lambda b: torch.stack([b, b + 99], dim=1)[:, 0], "float64": lambda b: b.double(), "int64": lambda b: b.long(),
         "float16": lambda b: b.half(), "column": lambda b: b[:, None], "grad": lambda b: b.clone().requires_grad_()}


@pytest.mark.parametrize("form", sorted(FORMS))
def test_levels_are_dense_float32_whatever_they_were(form):
    bins = torch.tensor([32.0, 16.0, 12.0])
    got = incoming._levels(FORMS[form](bins), 3, torch.device(DEV))
    assert got.dtype == torch.float32 and got.is_contiguous() and not got.requires_grad and torch.equal(got, bins)
    assert got.numpy().shape == (3,)
    with pytest.raises(RuntimeError, match="one entry per layer"):
        incoming._levels(FORMS[form](bins), 4, torch.device(DEV))


@pytest.mark.gpu
@pytest.mark.parametrize("device", ["cpu", DEV])
@pytest.mark.parametrize("form", sorted(FORMS))
def test_containers_take_levels_of_any_type_and_stride(form, device):
    from cachegen_amd import codec
    from cachegen_amd.kvgen import make_kv
    from cachegen_amd.serde import wire
    kb, vb = torch.tensor([32.0, 16.0, 12.0], device=device), torch.tensor([16.0, 8.0, 32.0], device=device)
    enc = codec.encode_kv(make_kv(3, 300, 2, 64, seed=5, device=DEV), kb.to(DEV), vb.to(DEV), chunk_tokens=256)
    want = codec.decode_encoded(enc, FORMS[form](kb), FORMS[form](vb), out_dtype=torch.float16)
    items, out = [], torch.zeros_like(want)
    for i, blob in enumerate(wire.pack_chunks(enc, compact=True)):
        items.append((incoming.Container.flat(blob), FORMS[form](kb), FORMS[form](vb), 256 * i))
    incoming.decode(items, out, "vllm")
    assert torch.equal(out.view(torch.int16), want.view(torch.int16))


def test_the_serializers_tables_follow_its_bins(monkeypatch):
    """The table size is that of the tensors a call codes with: what the hooks returned, what a program
    put in their place, and what it wrote into them."""
    from cachegen_amd import codec
    from cachegen_amd.config import LMCacheEngineConfig, LMCacheEngineMetadata
    from cachegen_amd.serde import cachegen_basics as basics
    from cachegen_amd.serde.cachegen_encoder import CacheGenSerializer
    taken = []

    def encode(kv, key_bins, value_bins, chunk_tokens=None, max_bins=None, **kw):
        taken.append(max_bins if max_bins is not None else codec._largest(key_bins, value_bins))
        raise KeyError
    monkeypatch.setattr(codec, "encode_kv", encode)
    monkeypatch.setattr(torch.Tensor, "cuda", lambda self: self)

    class Finer(CacheGenSerializer):
        def make_key_bins(self, config):
            return basics.make_key_bins(config) * 2

    def size(s):
        for call in (s.to_bytes, lambda kv: s.to_bytes_chunks(kv, 4)):
            with pytest.raises(KeyError):
                call(torch.zeros(32, 2, 8, 1, 8).half())
        assert taken[-1] == taken[-2]
        return taken[-1]
    for wire_format in ("pickle", "flat", "compact"):
        args = LMCacheEngineConfig.from_defaults(), LMCacheEngineMetadata("lmsys/longchat-7b-16k", 1, 0, "vllm"), wire_format
        assert size(CacheGenSerializer(*args)) == 32
        s = Finer(*args)
        assert size(s) == 64
        s.value_bins = torch.full((32,), 100.0)
        assert size(s) == 100
        s.value_bins[3] = 120
        assert size(s) == 120
        s.value_bins.fill_(8)
        assert size(s) == 64
        with torch.inference_mode():
            s.key_bins = torch.full((32,), 16.0)
            assert size(s) == 16
            s.key_bins[0] = 20
        assert size(s) == 20


@pytest.mark.gpu
def test_an_error_behind_a_launch_that_stores_to_the_host_is_waited_out(monkeypatch):
    """Writer and reader of compact containers, with something failing between the launch and the read."""
    import dataclasses
    from cachegen_amd import codec
    from cachegen_amd.kvgen import make_kv
    from cachegen_amd.serde import wire
    waited = []
    wait = hostmem.StoredWords._wait
    monkeypatch.setattr(hostmem.StoredWords, "_wait", lambda self: (waited.append(self.words.numel()), wait(self)))
    bins = torch.tensor([32.0, 16.0])
    enc = codec.encode_kv(make_kv(2, 256, 2, 64, seed=3, device=DEV), bins, bins)
    blob = wire.pack_chunks(enc, compact=True)[0]
    assert waited == [3 + 2 + 4]                             # status, wide, inexact, two boundaries, four rows' symbols
    with pytest.raises(AttributeError):
        wire.pack_chunks(dataclasses.replace(enc, maxima=types.SimpleNamespace(dtype=torch.float16)))
    assert waited == [9, 3 + 2]
    monkeypatch.setattr(codec, "decode_listed", lambda *a: {}["launch failed"])
    with pytest.raises(KeyError):
        incoming.decode([(incoming.Container.flat(blob), bins, bins, 0)], torch.empty((2, 2, 256, 2, 64), dtype=torch.float16, device=DEV), "vllm")
    assert waited == [9, 5, 1]
