"""The work that users of this codec have it do, as timed cases.

A case is a dict of plain values; `prepare` makes what a program holds before the call (a KV
cache, an encoded cache, blobs, an engine), `run` is one pass through the public entry points and
returns everything that pass computes.  KV caches come from `cachegen_amd.kvgen`: a standard
deviation per channel, a few outlier channels, values correlated along the tokens.

kind            what a pass is
--------------  --------------------------------------------------------------------------------
encode          codec.encode_kv over a whole cache; `keep`: with the workspace and result tensors of
                the call before (a serving loop), else with nothing but the cache and the bins in
                hand, checked, and the streams copied into the program's own buffer (a one-off call)
decode          codec.decode_encoded into a tensor that the program keeps
levels          codec.encode_kv_levels: one cache at several quantization levels
from_bytes      Deserializer.from_bytes of one chunk (flat containers)
round_trip      Serializer.to_bytes, then from_bytes, in any container
engine          LMCacheEngine.store of a context into a remote store, then retrive
merge           adaptive.merge: chunks at different levels decoded into one cache
entry_points    the reference extension's functions on one sub-chunk of symbols: table, streams,
                streams packed back to back, symbols again
"""
import math
import random

import torch

from cachegen_amd import adaptive, codec, torchac_hip
from cachegen_amd.cache_engine import LMCacheEngineBuilder
from cachegen_amd.config import LMCacheEngineConfig, LMCacheEngineMetadata
from cachegen_amd.kvgen import make_kv
from cachegen_amd.serde import CreateSerde
from cachegen_amd.serde.cachegen_basics import CacheGenConfig, CacheGenGPUBytestream, make_key_bins, make_value_bins
from cachegen_amd.serde.cachegen_decoder import decode_chunk
from cachegen_amd.serde.cachegen_encoder import encode_ntokens

# layers of the models whose bins tables the serializers know
MODELS = {"lmsys/longchat-7b-16k": 32, "Yukang/LongAlpaca-70B-16k": 80}
# bins of the key tiers and of the value tiers (CacheGenConfig.from_layer_tiers); "C" is the
# reference's level 2, "B" its level 1, "A" and "D" a coarser and a finer one
TIERS = {"A": ((8, 8, 8), (8, 8)), "B": ((16, 16, 12), (16, 12)),
         "C": ((32, 16, 16), (32, 16)), "D": ((64, 32, 32), (64, 32))}
DTYPES = {"float16": torch.float16, "bfloat16": torch.bfloat16}
DEVICE = "cuda:0"


def listed():
    return [
        # a 7B-shape context kept on the card, one table per 256 tokens: the headline benchmark
        dict(name="encode_context", kind="encode", layers=32, tokens=8192, heads=8, head_size=128, chunk=256,
             bins="C", dtype="float16", fmt="vllm", keep=True),
        dict(name="decode_context", kind="decode", layers=32, tokens=8192, heads=8, head_size=128, chunk=256,
             bins="C", dtype="float16", fmt="vllm"),
        # the largest: a 70B-shape context in 1500-token chunks (long-context streaming)
        dict(name="encode_long", kind="encode", layers=80, tokens=32768, heads=8, head_size=128, chunk=1500,
             bins="C", dtype="float16", fmt="vllm", keep=True),
        # a cache with all its heads (4096 channels), read back in the [head, token] layout
        dict(name="decode_wide", kind="decode", layers=32, tokens=16384, heads=32, head_size=128, chunk=256,
             bins="C", dtype="float16", fmt="huggingface"),
        # the smallest cache of the benchmark list, two sub-chunks under one table, nothing kept
        dict(name="encode_small", kind="encode", layers=2, tokens=512, heads=8, head_size=64, chunk=512,
             bins="C", dtype="bfloat16", fmt="huggingface", keep=False),
        # every level of an adaptive stream at once
        dict(name="encode_levels", kind="levels", layers=32, tokens=4096, heads=8, head_size=128, chunk=256,
             bins="ABCD", dtype="float16", fmt="vllm"),
        # what a store does with one chunk of the engine's default size: in and out, and out alone
        dict(name="chunk_round_trip", kind="round_trip", model="lmsys/longchat-7b-16k", tokens=256, heads=8, head_size=128,
             serde="cachegen-flat", dtype="bfloat16", fmt="vllm"),
        dict(name="chunk_from_bytes", kind="from_bytes", model="lmsys/longchat-7b-16k", tokens=256, heads=8, head_size=128,
             serde="cachegen-compact", dtype="bfloat16", fmt="vllm"),
        # the reference serializer's own call, a context that is no multiple of anything under one table
        dict(name="context_round_trip", kind="round_trip", model="lmsys/longchat-7b-16k", tokens=1333, heads=8, head_size=128,
             serde="cachegen", dtype="float16", fmt="huggingface"),
        # a prompt's cache put into and taken out of the remote store, the last chunk short
        dict(name="engine_context", kind="engine", model="lmsys/longchat-7b-16k", tokens=2100, heads=8, head_size=128, chunk=256,
             serde="cachegen-flat", dtype="bfloat16", fmt="vllm"),
        # the receiving end of an adaptive stream in the reference's 1500-token chunks
        dict(name="merge_stream", kind="merge", tokens=6000, heads=8, head_size=128, chunk=1500,
             dtype="float16", fmt="huggingface"),
        # the four functions of the reference's extension on a small model's sub-chunk
        dict(name="entry_points", kind="entry_points", layers=2, tokens=256, heads=8, head_size=64, bins="C", dtype="float16"),
    ]


def _log(rng, low, high):
    """A whole number between low and high, even over its logarithm."""
    return min(high, max(low, int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))))


def draw(rng: random.Random):
    kind = rng.choice(["encode", "encode", "decode", "decode", "levels", "from_bytes", "round_trip", "round_trip",
                       "engine", "merge", "entry_points"])
    c = dict(kind=kind)
    c["heads"], c["head_size"] = rng.choice([(8, 128), (8, 128), (32, 128), (8, 64), (4, 128), (5, 80), (12, 64), (16, 96)])
    channels = c["heads"] * c["head_size"]
    c["dtype"] = rng.choice(["float16", "bfloat16"])

    def tokens(layers, low, high, most_values):
        return _log(rng, low, max(low, min(high, most_values // (2 * layers * channels))))

    if kind in ("encode", "decode", "levels"):
        c["layers"] = _log(rng, 2, 80)
        c["tokens"] = tokens(c["layers"], 16, 32768, (1 << 28) if kind == "levels" else (1 << 30))
        c["chunk"] = rng.choice([256, 256, 1500, 512, _log(rng, 16, 2048), c["tokens"]])
        c["bins"] = "".join(sorted(rng.sample("ABCD", rng.randint(2, 4)))) if kind == "levels" else rng.choice("BCCD")
        c["fmt"] = rng.choice(["vllm", "huggingface"])
        if kind == "encode":
            c["keep"] = rng.random() < 0.7
    elif kind == "entry_points":
        c["layers"] = _log(rng, 1, 80)
        c["tokens"] = rng.randint(1, 256)
        c["bins"] = rng.choice("BCCD")
    elif kind == "merge":
        c["chunk"] = rng.choice([256, 1500, rng.randint(64, 1500)])
        c["tokens"] = tokens(32, c["chunk"], 8 * c["chunk"] + rng.randint(0, 63), 1 << 28)
        c["fmt"] = rng.choice(["vllm", "huggingface"])
    else:
        c["fmt"] = rng.choice(["vllm", "huggingface"])
        if kind == "engine":
            c["model"] = "lmsys/longchat-7b-16k"
            c["chunk"] = rng.choice([256, 256, rng.randint(64, 1024)])
            c["serde"] = rng.choice(["cachegen-flat", "cachegen-compact", "cachegen"])
        else:
            c["model"] = rng.choice(sorted(MODELS))
            c["serde"] = rng.choice(["cachegen-flat", "cachegen-compact"] + (["cachegen"] if kind == "round_trip" else []))
        c["tokens"] = tokens(MODELS[c["model"]], 16, 4096 if kind == "engine" else 2048, 1 << 28)
    return c


# ---- sizes ---------------------------------------------------------------------------------
def _layers(case):
    return case["layers"] if "layers" in case else MODELS.get(case.get("model"), 32)


def _bins(name, layers, device):
    """(key bins, value bins) with the reference's shares of the layers in every tier."""
    k, v = TIERS[name]
    first, second, vfirst = max(1, layers * 10 // 32), max(1, layers * 20 // 32), max(1, layers * 2 // 32)
    cfg = CacheGenConfig.from_layer_tiers(layers, [(first, k[0]), (second, k[1]), k[2]], [(vfirst, v[0]), v[1]])
    return make_key_bins(cfg).to(device), make_value_bins(cfg).to(device), max(k + v)


def work(case):
    """Bytes of one pass: the 16-bit cache, and what stands for it once encoded (streams of the
    measured size per symbol, tables, lengths, row maxima), each once per direction."""
    L, T, C = _layers(case), case["tokens"], case["heads"] * case["head_size"]
    n = 2 * L * T * C
    bits = {"A": 0.15, "B": 0.4, "C": 0.75, "D": 1.5}                  # per symbol
    kind = case["kind"]

    def encoded(level, chunk):
        nchunks = -(-T // chunk)
        nsub = (T // chunk) * -(-chunk // 256) + -(-(T % chunk) // 256)
        return n * bits[level] / 8 + 2 * L * C * (nchunks * 2 * (max(max(t) for t in TIERS[level]) + 1) + nsub * 4) + 4 * L * T

    if kind in ("encode", "decode"):
        b = 2 * n + encoded(case["bins"], case["chunk"])
    elif kind == "levels":
        b = 2 * n + sum(encoded(v, case["chunk"]) for v in case["bins"])
    elif kind == "from_bytes":
        b = 2 * n + encoded("C", T)
    elif kind == "round_trip":
        b = 2 * (2 * n + encoded("C", T))
    elif kind == "engine":
        b = 2 * (2 * n + encoded("C", case["chunk"]))
    elif kind == "merge":
        b = 2 * n + encoded("C", case["chunk"])
    else:
        n = L * 2 * T * C
        b = 3 * n + 2 * (n * bits[case["bins"]] / 8 + 2 * L * C * (2 * 33 + 4))
    return {"bytes": float(b), "flops": 0.0}


def tolerance(case):
    """Symbols, tables, streams and blobs are whole numbers; the dequantized values are defined to
    the bit by the same float32 steps in the same order."""
    return "exact"


# ---- states --------------------------------------------------------------------------------
def _cache(case, seed):
    L, T = _layers(case), case["tokens"]
    kv = make_kv(L, T, case["heads"], case["head_size"], seed=seed, device=DEVICE, dtype=DTYPES[case["dtype"]])
    if case.get("fmt") == "huggingface":
        kv = kv.permute(0, 1, 3, 2, 4).contiguous()
    return kv


def _engine(case):
    config = LMCacheEngineConfig(case["chunk"], None, "mem://contexts-%s:0" % case["serde"], case["serde"], False)
    metadata = LMCacheEngineMetadata(case["model"], 1, 0, case["fmt"])
    return LMCacheEngineBuilder.get_or_create("%s/%s/%d" % (case["serde"], case["fmt"], case["chunk"]), config, metadata)


def prepare(case, seed):
    kind = case["kind"]
    kv = _cache(case, seed)
    s = dict(case=case, kv=kv)
    if kind in ("encode", "decode", "entry_points"):
        kb, vb, top = _bins(case["bins"], case["layers"], DEVICE)
        s.update(kb=kb, vb=vb, max_bins=top)
    if kind == "encode" and not case["keep"]:
        nsub = codec.num_subchunks(case["tokens"], case["chunk"])
        s["sink"] = torch.zeros(nsub * 2 * kv[0, 0].numel() // case["tokens"] * case["layers"] * 256, dtype=torch.uint8, device=DEVICE)
    elif kind == "encode":
        s["workspace"] = torch.empty(codec.encode_workspace_bytes(case["layers"], case["tokens"], case["heads"] * case["head_size"],
                                                                  case["chunk"]), dtype=torch.uint8, device=DEVICE)
        s["out"] = codec.encode_kv(kv, kb, vb, chunk_tokens=case["chunk"], fmt=case["fmt"], max_bins=top, workspace=s["workspace"])
        s["out"].payload[s["out"].total_bytes():].zero_()        # the buffer is larger than the streams: its rest is never written
    elif kind == "decode":
        enc = codec.encode_kv(kv, kb, vb, chunk_tokens=case["chunk"], fmt=case["fmt"], max_bins=top)
        enc.payload = enc.payload[:enc.total_bytes()].clone()    # what arrives is the streams, without the buffer's rest
        s["enc"] = enc
        s["out"] = torch.empty_like(kv, dtype=torch.bfloat16 if case["fmt"] == "vllm" else torch.float16)
        del s["kv"]
    elif kind == "levels":
        tables = [_bins(v, case["layers"], DEVICE) for v in case["bins"]]
        s["levels"] = [t[:2] for t in tables]
        s["max_bins"] = [t[2] for t in tables]
        s["workspace"] = torch.empty(codec.encode_levels_workspace_bytes(case["layers"], case["tokens"], case["heads"] * case["head_size"],
                                                                         case["chunk"], len(tables)), dtype=torch.uint8, device=DEVICE)
        s["out"] = codec.encode_kv_levels(kv, s["levels"], chunk_tokens=case["chunk"], fmt=case["fmt"], max_bins=s["max_bins"],
                                          workspace=s["workspace"])
        for e in s["out"]:
            e.payload[e.total_bytes():].zero_()
    elif kind in ("from_bytes", "round_trip"):
        config = LMCacheEngineConfig.from_defaults(chunk_size=case["tokens"], remote_serde=case["serde"])
        s["ser"], s["de"] = CreateSerde(case["serde"], config, LMCacheEngineMetadata(case["model"], 1, 0, case["fmt"]))
        if kind == "from_bytes":
            s["blob"] = s["ser"].to_bytes(kv)
            del s["kv"]
    elif kind == "engine":
        s["engine"] = _engine(case)
        s["tokens"] = torch.randint(0, 32000, [case["tokens"]], generator=torch.Generator().manual_seed(seed))
        s["kv"] = tuple((layer[0], layer[1]) for layer in torch.unbind(kv, dim=0))
    elif kind == "merge":
        # chunks are sent at the level their bandwidth allows; one of them is recomputed instead
        rng = random.Random(seed)
        s["blobs"] = adaptive.encode_levels(kv, case["chunk"], fmt=case["fmt"])
        s["configs"] = [rng.choice((1, 2, 3)) for _ in s["blobs"]]
        if len(s["configs"]) > 1:
            s["configs"][rng.randrange(len(s["configs"]))] = 0
    elif kind == "entry_points":
        sym, _ = codec.quantize_kv(kv, s["kb"], s["vb"])
        rows, T, C = sym.shape
        s["sym"] = sym.view(torch.int8)
        s["buffer"] = torch.zeros((rows, C, 256), dtype=torch.uint8, device=DEVICE)
        s["lengths"] = torch.zeros((rows, C), dtype=torch.int32, device=DEVICE)
        s["decoded"] = torch.zeros((rows, T, C), dtype=torch.uint8, device=DEVICE)
        del s["kv"]
    return s


def _fields(enc, payload):
    return {"cdf": enc.cdf, "maxima": enc.maxima, "lengths": enc.lengths, "offsets": enc.offsets, "payload": payload, "status": enc.status}


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "encode":
        if case["keep"]:
            enc = codec.encode_kv(state["kv"], state["kb"], state["vb"], chunk_tokens=case["chunk"], fmt=case["fmt"],
                                  max_bins=state["max_bins"], workspace=state["workspace"], out=state["out"])
            return _fields(enc, enc.payload)
        enc = codec.encode_kv(state["kv"], state["kb"], state["vb"], chunk_tokens=case["chunk"], fmt=case["fmt"])
        enc.check()
        n = enc.total_bytes()
        state["sink"][:n].copy_(enc.payload[:n])
        return _fields(enc, state["sink"])
    if kind == "decode":
        return codec.decode_encoded(state["enc"], state["kb"], state["vb"], fmt=case["fmt"], out=state["out"])
    if kind == "levels":
        encs = codec.encode_kv_levels(state["kv"], state["levels"], chunk_tokens=case["chunk"], fmt=case["fmt"],
                                      max_bins=state["max_bins"], workspace=state["workspace"], out=state["out"])
        return [_fields(e, e.payload) for e in encs]
    if kind == "from_bytes":
        return state["de"].from_bytes(state["blob"])
    if kind == "round_trip":
        return state["de"].from_bytes(state["ser"].to_bytes(state["kv"]))
    if kind == "engine":
        state["engine"].store(state["tokens"], state["kv"], skip_existing=False)
        kv, _ = state["engine"].retrive(state["tokens"])
        return kv
    if kind == "merge":
        return adaptive.merge(state["configs"], state["blobs"], case["chunk"], case["tokens"], orig_kv=state["kv"], fmt=case["fmt"])
    cdf = torchac_hip.calculate_cdf(state["sym"], state["max_bins"])
    stream = encode_ntokens(cdf, state["sym"], state["buffer"], state["lengths"])
    decode_chunk(cdf, CacheGenGPUBytestream(stream, state["lengths"], state["sym"].shape[1]), state["decoded"])
    return {"cdf": cdf, "streams": state["buffer"], "lengths": state["lengths"], "symbols": state["decoded"]}
