"""CacheGenDeserializer on MI355X
(LMCache/lmcache/storage_backend/serde/cachegen_decoder.py in the reference)."""
from typing import List

import torch

from .. import codec, torchac_hip
from ..config import LMCacheEngineConfig, LMCacheEngineMetadata
from . import cachegen_basics as CGBasics
from . import incoming, pickled, wire
from .cachegen_basics import CacheGenConfig, CacheGenGPUBytestream, CacheGenGPUEncoderOutput
from .serde import Deserializer


def decode_chunk(cdf: torch.Tensor, data_chunk: CacheGenGPUBytestream, target_buffer: torch.Tensor):
    """cachegen_decoder.py:52-75: decode one sub-chunk's streams into
    target_buffer [2L, ntokens, nchannels] (a strided view is fine)."""
    torchac_hip.decode_fast_lengths(cdf, data_chunk.bytestream, data_chunk.bytestream_lengths, target_buffer)


def decode_function_gpu(cdf: torch.Tensor, data_chunks: List[CacheGenGPUBytestream],
                        layers_in_key: int, chunk_size: int, output: torch.Tensor):
    """cachegen_decoder.py:77-112: symbols of every sub-chunk -> (key, value) float32
    [layers_in_key, chunk_size, nchannels]."""
    nlayers, nchannels, _ = cdf.shape
    output = output.reshape((nlayers, chunk_size, nchannels))
    start = 0
    for data_chunk in data_chunks:
        end = start + data_chunk.ntokens
        decode_chunk(cdf, data_chunk, output[:, start:end, :])
        start = end
    out = output.reshape((2, layers_in_key, chunk_size, nchannels))
    key, value = out.float()
    return key, value


def do_dequantize(t: torch.Tensor, bins: torch.Tensor, maxtensors: torch.Tensor):
    """cachegen_decoder.py:24-34 (plain tensor ops; the fused path does this in-kernel)."""
    C = (bins // 2 - 1)[:, None, None]
    t = t - C
    t = t / C
    t = t * maxtensors
    return t


class CacheGenDeserializer(Deserializer):
    def __init__(self, config: LMCacheEngineConfig, metadata: LMCacheEngineMetadata):
        self.cachegen_config = CacheGenConfig.from_model_name(metadata.model_name)
        self.chunk_size = config.chunk_size
        self.fmt = metadata.fmt
        self.key_bins = self.make_key_bins(self.cachegen_config)
        self.value_bins = self.make_value_bins(self.cachegen_config)

    def make_key_bins(self, config: CacheGenConfig) -> torch.Tensor:
        return CGBasics.make_key_bins(config).cuda()

    def make_value_bins(self, config: CacheGenConfig) -> torch.Tensor:
        return CGBasics.make_value_bins(config).cuda()

    def from_bytes(self, bs: bytes) -> torch.Tensor:
        """Returns bfloat16 [num_layers, 2, num_tokens, num_heads, head_size] for fmt "vllm",
        float16 [num_layers, 2, num_heads, num_tokens, head_size] for "huggingface"
        (cachegen_decoder.py:144-173).  Decode, dequantization, cast and layout are one
        kernel.  Blobs in the flat container of `wire` are recognised by their magic."""
        return self._decode(bs, None)

    def from_bytes_into(self, bs: bytes, out: torch.Tensor) -> torch.Tensor:
        """Decodes `bs` straight into `out`: a tensor, or a view into a larger one, of the
        chunk's shape in this deserializer's layout, float16 or bfloat16 (not in the reference,
        whose callers concatenate the decoded chunks)."""
        return self._decode(bs, out)

    def chunk_shape(self, bs: bytes):
        """Shape `from_bytes(bs)` would have, read from a flat container's header without
        decoding; None for a pickle container."""
        if not wire.is_flat(bs):
            return None
        h = wire.read_header(bs)
        L, T, H, D = h["num_layers"], h["num_tokens"], h["num_heads"], h["head_size"]
        return (L, 2, T, H, D) if self.fmt == "vllm" else (L, 2, H, T, D)

    def _decode(self, bs, out):
        if wire.is_flat(bs):
            return self._from_container(incoming.Container.flat(bs), out)
        container = pickled.container(bs)
        if container is not None:
            try:
                return self._from_container(container, out)
            except incoming.LengthsError:
                pass                             # lengths that are not the stored streams': decoded as they say, below
        encoder_output = CacheGenGPUEncoderOutput.from_bytes(bs)
        cdf = encoder_output.cdf.cuda()
        max_k = encoder_output.max_tensors_key.cuda()
        max_v = encoder_output.max_tensors_value.cuda()
        nlayers, ntokens = max_k.shape[0], max_k.shape[1]
        chunks = encoder_output.data_chunks
        if len(chunks) == 1:
            payload = chunks[0].bytestream.cuda()
            lengths = chunks[0].bytestream_lengths.cuda()
        else:
            payload = torch.cat([c.bytestream.cuda() for c in chunks])
            lengths = torch.stack([c.bytestream_lengths.cuda() for c in chunks])
        offsets = codec.scan_lengths(lengths)
        maxima = torch.stack([max_k.reshape(nlayers, ntokens), max_v.reshape(nlayers, ntokens)])
        return codec.decode_kv(cdf.unsqueeze(0), maxima, offsets, payload, self.key_bins,
                               self.value_bins, nlayers, ntokens, encoder_output.num_heads,
                               encoder_output.head_size, chunk_tokens=ntokens, fmt=self.fmt, out=out)

    def _from_container(self, container, out=None) -> torch.Tensor:
        L, T, H, D = container.num_layers, container.num_tokens, container.num_heads, container.head_size
        self._check_layers(container)
        if out is None:
            shape = (L, 2, T, H, D) if self.fmt == "vllm" else (L, 2, H, T, D)
            out = torch.empty(shape, dtype=torch.bfloat16 if self.fmt == "vllm" else torch.float16, device=self.key_bins.device)
        elif out.shape[2 if self.fmt == "vllm" else 3] != T:
            raise RuntimeError("output tensor does not match the encoded geometry")
        return incoming.decode([(container, self.key_bins, self.value_bins, 0)], out, self.fmt)

    def _check_layers(self, container):
        if container.num_layers != self.key_bins.numel():
            raise ValueError("blob has %d layers, this deserializer's model %d"
                             % (container.num_layers, self.key_bins.numel()))

    def from_bytes_concat(self, blobs: List[bytes]):
        """The tensors of several blobs side by side along the token dimension, in one tensor that
        they are decoded into by one launch; None if that takes the blobs one by one (not in the
        reference, whose callers concatenate the decoded chunks)."""
        items, tokens = [], 0
        for bs in blobs:
            container = incoming.Container.flat(bs) if wire.is_flat(bs) else pickled.container(bs)
            if container is None:
                return None
            self._check_layers(container)
            items.append((container, self.key_bins, self.value_bins, tokens))
            tokens += container.num_tokens
        first = items[0][0]
        L, H, D = first.num_layers, first.num_heads, first.head_size
        shape = (L, 2, tokens, H, D) if self.fmt == "vllm" else (L, 2, H, tokens, D)
        out = torch.empty(shape, dtype=torch.bfloat16 if self.fmt == "vllm" else torch.float16, device=self.key_bins.device)
        try:
            return incoming.decode(items, out, self.fmt)
        except incoming.LengthsError:
            return None
