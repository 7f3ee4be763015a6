"""The workloads this library is measured on, each through a public entry point.

A case is a dict of plain values.  `kind` names the call:

  object     one memory object <-> paged caches (multi_layer_kv_transfer), the
             connector's call per chunk; in device or pinned host memory
  batch      all memory objects of a request in one call
             (multi_layer_kv_transfer_batched), K/V or MLA latent caches
  layer      one layer of the caches (single_layer_kv_transfer), the layerwise
             connector's call
  encode     CacheGen compression of a chunk's symbols (formats.encode_chunk)
  decode     the chunk back to symbols (formats.decode_chunk)
  roundtrip  both, one after the other
  rope       K re-rotation of a reused prefix (rotary_embedding_k_fused)
  sparse     decode-time copy of the selected tokens of an MLA layer into the
             device caches (sparse_graph_kv_transfer)
"""

import math
import os
import sys

import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "lmcache-ascend_amd"))

from lmcache_amd import c_ops, formats  # noqa: E402

CHUNK = 256  # tokens per memory object
MLA_K, MLA_PE = 512, 64  # latent and rope columns of an MLA cache row
DTYPES = {"bf16": torch.bfloat16, "f16": torch.float16}


def _object(name, store, layers, width, block, tokens, host=False, pad=0.0):
    return {"name": name, "kind": "object", "store": store, "layers": layers, "width": width, "block": block,
            "tokens": tokens, "host": host, "pad": pad, "mla": False, "dtype": "bf16"}


def _batch(name, store, layers, width, block, tokens, pad=0.0, mla=False):
    return dict(_object(name, store, layers, width, block, tokens, False, pad), kind="batch", mla=mla)


def _codec(name, kind, planes, tokens, channels, bins=32):
    return {"name": name, "kind": kind, "planes": planes, "tokens": tokens, "channels": channels, "bins": bins}


def listed():
    return [
        # The smallest call: one 16-token block of a 4-layer cache (the CPU
        # plumbing shape), stored by itself.  Latency and the launch count.
        _object("store_one_block", True, 4, 1024, 16, 16),
        # A 4096-token batch of an 8-KV-head, 32-layer model stored in one
        # call: the headline shape.
        _batch("store_batch_32l", True, 32, 1024, 128, 4096),
        # A long prefix of a 64-layer model loaded back, 5% of its slots
        # padding: the largest transfer.
        _batch("retrieve_batch_64l_padded", False, 64, 1024, 128, 8192, pad=0.05),
        # One rank of a TP-8, 80-layer model (one KV head, 256-byte rows): a
        # request's ragged last object, loaded by its own call.
        _object("retrieve_object_tp8_ragged", False, 80, 128, 64, 199),
        # MLA latent caches (576 columns, 61 layers): a 16384-token prefill
        # stored.
        _batch("store_batch_mla", True, 61, MLA_K + MLA_PE, 64, 16384, mla=True),
        # The layerwise connector's call: one layer's 4096 tokens into its
        # paged caches.
        dict(_object("retrieve_layer", False, 1, 1024, 128, 4096), kind="layer"),
        # Offload to the CPU: one 256-token object stored to pinned memory
        # over PCIe.
        _object("store_object_pinned", True, 32, 1024, 128, 256, host=True),
        # CacheGen: one 256-token chunk of K and V of 32 layers, compressed.
        _codec("encode_chunk", "encode", 64, 256, 1024),
        # The same chunk on its way back.
        _codec("decode_chunk", "decode", 64, 256, 1024),
        # A long, odd chunk of a 28-layer model's TP slice (two heads).
        _codec("roundtrip_long_chunk", "roundtrip", 56, 1000, 256),
        # Blending: 4096 reused K rows of 8 heads moved to new positions.
        {"name": "rope_prefix", "kind": "rope", "tokens": 4096, "heads": 8, "dim": 128, "neox": True, "dtype": "bf16"},
        # Sparse attention's decode step: 2048 selected tokens of each of 64
        # requests gathered from device chunks.
        {"name": "sparse_decode", "kind": "sparse", "requests": 64, "selected": 2048, "limit": 8192},
    ]


def _log(rng, lo, hi):
    """A whole number in [lo, hi], even over its logarithm."""
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi + 1)))))))


def draw(rng):
    kind = rng.choice(["object", "pinned", "batch", "mla", "layer", "encode", "decode", "roundtrip", "rope", "sparse"])
    store = rng.random() < 0.5
    pad = rng.choice([0.0, 0.05])
    # KV width of one rank: 1 to 8 heads.
    width = rng.randint(1, 8) * rng.choice([64, 96, 128])
    block = rng.choice([16, 64, 128])
    if kind in ("object", "pinned"):
        c = _object("", store, rng.choice([4, 28, 32, 64, 80]), width, block, _log(rng, 1, CHUNK), kind == "pinned", pad)
    elif kind == "batch":
        c = _batch("", store, rng.choice([4, 28, 32, 64]), width, block, _log(rng, CHUNK + 1, 8192), pad)
    elif kind == "mla":
        c = _batch("", store, rng.choice([4, 27, 61]), MLA_K + MLA_PE, 64, _log(rng, 1, 16384), pad, True)
    elif kind == "layer":
        c = dict(_object("", store, 1, width, block, _log(rng, 1, 32768), False, pad), kind="layer")
    elif kind in ("encode", "decode", "roundtrip"):
        tokens = _log(rng, 1, 1024)
        # One rank's channels, in whole groups of 32 as the decoder takes them.
        channels = rng.randint(1, 8) * rng.choice([64, 96, 128])
        planes = 2 * _log(rng, 1, max(1, min(64, (64 * 256 * 1024) // (2 * tokens * channels))))
        c = _codec("", kind, planes, tokens, channels, rng.choice([16, 32, 32]))
    elif kind == "rope":
        c = {"kind": "rope", "tokens": _log(rng, 1, 16384), "heads": rng.randint(1, 8), "dim": rng.choice([64, 96, 128]),
             "neox": rng.random() < 0.75, "dtype": rng.choice(["bf16", "bf16", "f16"])}
    else:
        c = {"kind": "sparse", "requests": _log(rng, 1, 64), "selected": _log(rng, 64, 2048), "limit": rng.choice([2048, 4096, 8192])}
    c.pop("name", None)
    return c


# ---------------------------------------------------------------------------
# Inputs
# ---------------------------------------------------------------------------


def prepare(case, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    make = {"object": _kv, "batch": _kv, "layer": _kv, "encode": _symbols_state, "decode": _decode_state,
            "roundtrip": _symbols_state, "rope": _rope_state, "sparse": _sparse_state}
    return dict(make[case["kind"]](case, gen), case=case)


def _kv(case, gen):
    """Paged caches of N(0, 1) rows, blocks handed out in random order to one
    request, its last block partly filled; memory objects of 256 tokens."""
    T, L, W, BS = case["tokens"], case["layers"], case["width"], case["block"]
    dt = DTYPES[case["dtype"]]
    planes = 1 if case["mla"] else 2
    used = -(-T // BS)
    blocks = 2 * used + 1
    order = torch.randperm(blocks, generator=gen, device="cuda")[:used]
    slots = (order[:, None] * BS + torch.arange(BS, device="cuda")).reshape(-1)[:T].contiguous()
    if case["pad"]:
        drop = torch.rand(T, generator=gen, device="cuda") < case["pad"]
        slots = torch.where(drop, torch.full_like(slots, -1), slots)
    shape = (L, planes, blocks, BS, W)
    if case["store"]:
        pool = torch.randn(shape, generator=gen, device="cuda", dtype=dt)
    else:
        pool = torch.zeros(shape, device="cuda", dtype=dt)
    # One tensor per layer and plane, as an engine keeps them; the library
    # takes their addresses.
    step = pool.stride(1) * pool.element_size()
    ptrs = torch.arange(L * planes, device="cuda", dtype=torch.int64) * step + pool.data_ptr()
    sizes = [T] if case["kind"] != "batch" else [min(CHUNK, T - s) for s in range(0, T, CHUNK)]
    objs = []
    for n in sizes:
        shape = (planes, n, W) if case["kind"] == "layer" else (planes, L, n, W)
        if case["store"]:
            o = torch.zeros(shape, dtype=dt, device="cuda")
        else:
            o = torch.randn(shape, generator=gen, dtype=dt, device="cuda")
        if case["host"]:
            h = torch.empty(shape, dtype=dt, pin_memory=True)
            h.copy_(o)
            o = h
        objs.append(o)
    return {"pool": pool, "ptrs": ptrs, "slots": slots, "objs": objs, "starts": list(range(0, T, CHUNK)),
            "caches": (pool[0, 0].view(blocks, BS, 1, W), pool[0, -1].view(blocks, BS, 1, W)), "rows": blocks * BS}


def _symbols(case, gen):
    """N(0, 1) keys and values quantised per channel, as the CacheGen serde
    does: the first 10 K layers to the full bin count, the others to 16.  The
    seed orders the channels of each plane and the tokens of each channel of
    one such chunk, so chunks of one case compress to the same size."""
    P, T, C = case["planes"], case["tokens"], case["channels"]
    x = torch.randn((P, T, C), generator=torch.Generator(device="cuda").manual_seed(T * C + P), device="cuda")
    bins = torch.full((P, 1, 1), 16.0, device="cuda")
    bins[: min(10, P // 2)] = case["bins"]
    half = torch.floor(bins / 2) - 1
    top = x.abs().amax(dim=1, keepdim=True).clamp_min(1e-30)
    symbols = (torch.round(x / top * half) + half).to(torch.uint8)
    channel = torch.rand((P, 1, C), generator=gen, device="cuda").argsort(dim=2)
    token = torch.rand((P, T, C), generator=gen, device="cuda").argsort(dim=1)
    return symbols.gather(2, channel.expand(P, T, C)).gather(1, token).contiguous()


def _symbols_state(case, gen):
    return {"symbols": _symbols(case, gen)}


def _decode_state(case, gen):
    return {"chunk": formats.encode_chunk(_symbols(case, gen), case["bins"])}


def _rope_state(case, gen):
    dt, D = DTYPES[case["dtype"]], case["dim"]
    n = case["tokens"]
    inv = 1.0 / (500000.0 ** (torch.arange(0, D, 2, dtype=torch.float32, device="cuda") / D))
    ang = torch.outer(torch.arange(n + 1000, dtype=torch.float32, device="cuda"), inv)
    old = torch.arange(n, dtype=torch.int64, device="cuda")
    return {"key": torch.randn((n, case["heads"] * D), generator=gen, device="cuda").to(dt),
            "cache": torch.cat((ang.cos(), ang.sin()), dim=-1).to(dt), "old": old, "new": old + 1000}


def _sparse_state(case, gen):
    """Each request's tokens in 256-token device chunks; its selected tokens
    go to distinct random slots of the caches."""
    R, S, limit, bs = case["requests"], case["selected"], case["limit"], 64
    S = min(S, limit)
    per = limit // CHUNK
    blocks = 2 * (-(-R * S // bs))
    k = torch.zeros((blocks, bs, 1, MLA_K), dtype=torch.bfloat16, device="cuda")
    pe = torch.zeros((blocks, bs, 1, MLA_PE), dtype=torch.bfloat16, device="cuda")
    src_k = torch.randn((R * per, CHUNK, MLA_K), generator=gen, dtype=torch.bfloat16, device="cuda")
    src_pe = torch.randn((R * per, CHUNK, MLA_PE), generator=gen, dtype=torch.bfloat16, device="cuda")
    at = torch.arange(R * per, dtype=torch.int64, device="cuda")
    table = torch.stack([src_k.data_ptr() + at * (CHUNK * MLA_K * 2), src_pe.data_ptr() + at * (CHUNK * MLA_PE * 2)])
    picked = torch.rand((R, limit), generator=gen, device="cuda").argsort(dim=1)[:, :S].to(torch.int32).contiguous()
    slots = torch.randperm(blocks * bs, generator=gen, device="cuda")[: R * S].reshape(R, S).contiguous()
    dest = c_ops.prepare_sparse_direct_destination_state((k, pe), slots, 5, 0, 0, 0)
    return {"k": k, "pe": pe, "sources": (src_k, src_pe), "table": table, "picked": picked, "slots": slots, "dest": dest,
            "counts": torch.full((R,), S, dtype=torch.int32, device="cuda"),
            "limits": torch.full((R,), limit, dtype=torch.int32, device="cuda")}


# ---------------------------------------------------------------------------
# One pass
# ---------------------------------------------------------------------------


def _chunk_out(chunk):
    return {"cdf": chunk.cdf, "lengths": chunk.lengths, "streams": chunk.streams}


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "encode":
        return _chunk_out(formats.encode_chunk(state["symbols"], case["bins"]))
    if kind == "decode":
        return formats.decode_chunk(state["chunk"])
    if kind == "roundtrip":
        chunk = formats.encode_chunk(state["symbols"], case["bins"])
        return dict(_chunk_out(chunk), symbols=formats.decode_chunk(chunk))
    if kind == "rope":
        c_ops.rotary_embedding_k_fused(state["old"], state["new"], state["key"], case["dim"], state["cache"], case["neox"])
        return state["key"]
    if kind == "sparse":
        c_ops.sparse_graph_kv_transfer(state["dest"], state["slots"], state["picked"], state["counts"], state["table"],
                                       state["limits"], CHUNK)
        return [state["k"], state["pe"]]
    device = state["slots"].device
    if kind == "layer":
        c_ops.single_layer_kv_transfer(state["objs"][0], state["caches"], state["slots"], case["store"], 2)
    elif kind == "object":
        c_ops.multi_layer_kv_transfer(state["objs"][0], state["ptrs"], state["slots"], device, state["rows"],
                                      case["store"], False, 2)
    else:
        c_ops.multi_layer_kv_transfer_batched(state["objs"], state["ptrs"], state["slots"], state["starts"], device,
                                              state["rows"], case["store"], case["mla"], 2)
    return state["objs"] if case["store"] else state["pool"]


# ---------------------------------------------------------------------------
# What a pass cannot do without, and what its outputs may differ by
# ---------------------------------------------------------------------------


def work(case):
    kind = case["kind"]
    if kind in ("encode", "decode", "roundtrip"):
        streams = case["planes"] * case["channels"]
        symbols = streams * case["tokens"]
        # Symbols; the CDF, the lengths and the streams (about 3.5 bits a
        # symbol) on the other side.
        one = symbols + streams * (2 * (case["bins"] + 1) + 4) + symbols * 3.5 / 8
        return {"bytes": one * (2 if kind == "roundtrip" else 1), "flops": 0}
    if kind == "rope":
        pairs = case["tokens"] * case["heads"] * case["dim"] // 2
        return {"bytes": 2 * 2 * 2 * pairs + case["tokens"] * (16 + 4 * case["dim"]), "flops": 12 * pairs}
    if kind == "sparse":
        n = case["requests"] * min(case["selected"], case["limit"])
        return {"bytes": n * (2 * 2 * (MLA_K + MLA_PE) + 12), "flops": 0}
    planes = 1 if case["mla"] else 2
    tokens = case["tokens"] * (1 - case["pad"])
    return {"bytes": 2 * 2 * planes * case["layers"] * tokens * case["width"] + 8 * case["tokens"], "flops": 0}


def tolerance(case):
    if case["kind"] != "rope":
        return "exact"  # copies, code tables, bitstreams and symbols
    # One rounding to the key's type; another order of the sums moves a
    # result by one place where it lies between two.
    return {"rel": 2e-3, "max": 1.6e-2} if case["dtype"] == "bf16" else {"rel": 2.5e-4, "max": 2e-3}


def exact(case, seed):
    """The re-rotated keys in 64 bits; the other cases move or code whole
    values."""
    if case["kind"] != "rope":
        return None
    s = prepare(case, seed)
    D, half = case["dim"], case["dim"] // 2
    x = s["key"].double().view(case["tokens"], case["heads"], D)
    cache = s["cache"].double()

    def angle(pos):
        row = cache[pos].unsqueeze(1)
        return row[..., :half], row[..., half:]

    if case["neox"]:
        a, b = x[..., :half], x[..., half:]
    else:
        a, b = x[..., 0::2], x[..., 1::2]
    c, n = angle(s["old"])
    a, b = a * c + b * n, b * c - a * n
    c, n = angle(s["new"])
    a, b = a * c - b * n, b * c + a * n
    out = torch.cat((a, b), dim=-1) if case["neox"] else torch.stack((a, b), dim=-1).flatten(-2)
    return out.reshape(case["tokens"], case["heads"] * D)
