"""GPU tests of the chunk codec's own paths (formats.encode_chunk and
decode_chunk) against the CPU oracle, at the sizes where their kernels can go
wrong: blocks of 64 streams that span layers or are partly filled, rows that
do not start on a dword, streams cut to a row's capacity, and chunks longer
than one 256-token piece."""

import numpy as np
import pytest
import torch

from oracle import cachegen as oc

pytestmark = pytest.mark.gpu

DEV = "cuda:0"


@pytest.fixture(scope="module")
def F():
    from lmcache_amd import formats

    return formats


def _symbols(L, T, C, nb, seed, kind="normal"):
    rng = np.random.default_rng(seed)
    if kind == "normal":
        return oc.quantize(rng.normal(0, 2, size=(L, T, C)).astype(np.float32), nb)
    if kind == "constant":  # one present symbol per stream: 1-bit codes
        return np.broadcast_to(rng.integers(0, nb, size=(L, 1, C), dtype=np.uint8), (L, T, C)).copy()
    # Skewed counts (the longest codes), with symbols past nb that are not coded.
    p = 0.5 ** np.minimum(np.arange(nb + 1), 14)
    return rng.choice(nb + 1, size=(L, T, C), p=p / p.sum()).astype(np.uint8)


# Streams end inside a block (L * C % 64 != 0), blocks span layers (C = 96,
# 32, 17), rows start at odd addresses (cap odd), and caps cut streams.
@pytest.mark.parametrize("kind", ["normal", "constant", "skewed"])
@pytest.mark.parametrize("L,T,C,nb,cap", [
    (1, 1, 32, 16, 0), (2, 256, 96, 32, 0), (3, 37, 17, 16, 0), (5, 255, 48, 32, 511), (3, 64, 96, 33, 7),
    (2, 257, 64, 32, 0), (1, 1000, 160, 32, 0), (2, 600, 33, 16, 301), (3, 300, 96, 64, 0), (1, 9, 1, 2, 0),
])
def test_encode_chunk_vs_oracle(F, L, T, C, nb, cap, kind):
    sym = _symbols(L, T, C, nb, L * T + C + nb, kind)
    chunk = F.encode_chunk(torch.from_numpy(sym).to(DEV), nb, cap)
    cdf = oc.calculate_cdf(sym, nb)
    rows, lens = oc.encode(cdf, sym, cap or 2 * T)
    kept = np.minimum(lens, rows.shape[2])
    want = np.concatenate([rows[l, c, :kept[l, c]] for l in range(L) for c in range(C)])
    assert np.array_equal(chunk.cdf.cpu().numpy(), cdf)
    assert np.array_equal(chunk.lengths.cpu().numpy(), lens)
    assert np.array_equal(chunk.streams.cpu().numpy(), want)


def test_encode_chunk_without_tokens_or_streams(F):
    for shape in [(2, 0, 64), (0, 5, 64), (2, 5, 0)]:
        chunk = F.encode_chunk(torch.zeros(shape, dtype=torch.uint8, device=DEV), 16)
        assert chunk.streams.numel() == 0
        assert chunk.lengths.shape == (shape[0], shape[2]) and int(chunk.lengths.sum()) == 0


@pytest.mark.parametrize("kind", ["normal", "constant", "skewed"])
@pytest.mark.parametrize("L,T,C,nb", [
    (1, 1, 32, 16), (1, 255, 96, 32), (3, 256, 160, 32), (1, 257, 32, 32), (2, 288, 96, 16), (3, 1000, 32, 32),
    (1, 1023, 64, 32), (5, 289, 96, 31), (1, 4097, 64, 32), (3, 300, 96, 48),
])
def test_chunk_round_trip(F, L, T, C, nb, kind):
    sym = np.minimum(_symbols(L, T, C, nb, T + C + nb, kind), nb - 1).astype(np.uint8)
    chunk = F.encode_chunk(torch.from_numpy(sym).to(DEV), nb)
    assert np.array_equal(F.decode_chunk(chunk).cpu().numpy(), sym)


# Rows that calculate_cdf does not make (long codes anywhere, bases off their
# place, zero-length codes) over random streams, some of them short of their
# symbols, at lengths around the decoder's epochs.
@pytest.mark.parametrize("T", [257, 260, 287, 288, 289, 1000])
@pytest.mark.parametrize("kind", ["codes", "sorted", "random"])
def test_decode_long_foreign_rows(kind, T):
    from lmcache_amd import c_ops

    L, C, nb = 3, 96, 32
    rng = np.random.default_rng(T + len(kind))
    if kind == "codes":
        sym = _symbols(L, 700, C, nb, T, "skewed")
        cdf = oc.calculate_cdf(np.minimum(sym, nb - 1).astype(np.uint8), nb)
    elif kind == "sorted":
        base = np.sort(rng.integers(0, 4096, size=(L, C, nb + 1)) * 16, axis=2)
        cdf = (base | rng.integers(0, 16, size=base.shape)).astype(np.uint16).view(np.int16)
    else:
        cdf = rng.integers(0, 65536, size=(L, C, nb + 1)).astype(np.uint16).view(np.int16)
    lens = rng.integers(0, T, size=(L, C)).astype(np.int32)
    prefix = np.cumsum(lens.reshape(-1), dtype=np.int64).astype(np.int32).reshape(L, C)
    stream = rng.integers(0, 256, size=int(prefix[-1, -1]), dtype=np.uint8)
    want = oc.decode(cdf, stream, prefix, T)
    out = torch.full((L, T, C), 255, dtype=torch.uint8, device=DEV)
    c_ops.decode_fast_prefsum(torch.from_numpy(cdf).to(DEV), torch.from_numpy(stream).to(DEV),
                              torch.from_numpy(prefix).to(DEV), out)
    assert np.array_equal(out.cpu().numpy(), want)


# Rows of codes of up to 8 bits, which the group cursor takes from per-lane
# regions: calculated codes, rows with a symbol 31 of length 8 (its entry reads
# as an escape) and random rows of that form (zero-length codes, gaps, wraps),
# streams that fit the regions and that do not, one kernel and the other, and
# blocks of 32 streams.
@pytest.mark.parametrize("L,C,T", [(3, 96, T) for T in (257, 384, 385, 1000, 1024, 1025)] + [(16, 1056, 257), (16, 1056, 385)])
@pytest.mark.parametrize("kind,nb", [("codes", 32), ("codes", 17), ("last", 32), ("random", 32), ("random", 9)])
def test_decode_long_short_codes(kind, nb, L, C, T):
    from lmcache_amd import c_ops

    rng = np.random.default_rng(T + nb + L)
    if kind == "codes":
        sym = rng.integers(0, min(nb, 12), size=(L, 200, C)).astype(np.uint8)
        cdf = oc.calculate_cdf(sym, nb)
    elif kind == "last":
        row = np.concatenate([[1], (0x8000 + 256 * np.arange(31)) | 8, [0]]).astype(np.uint16)
        cdf = np.broadcast_to(row.view(np.int16), (L, C, nb + 1)).copy()
    else:
        base = rng.integers(0, 256, size=(L, C, nb + 1)) << 8
        base[:, ::2] = np.sort(base[:, ::2], axis=2)
        base[:, 1::7] = 0
        cdf = (base | rng.integers(0, 9, size=base.shape)).astype(np.uint16).view(np.int16)
    # Neither the rows nor the streams start on a 16-byte boundary.
    held_cdf = torch.empty(cdf.size + 8, dtype=torch.int16, device=DEV)[T % 8:][:cdf.size].view(L, C, nb + 1)
    held_cdf.copy_(torch.from_numpy(cdf))
    for most in (T // 2, 3000) if L * C < 4096 else (T // 2,):
        lens = rng.integers(0, most, size=(L, C)).astype(np.int32)
        prefix = np.cumsum(lens.reshape(-1), dtype=np.int64).astype(np.int32).reshape(L, C)
        stream = rng.integers(0, 256, size=int(prefix[-1, -1]), dtype=np.uint8)
        want = oc.decode(cdf, stream, prefix, T)
        held = torch.full((stream.size + 16,), 0xFF, dtype=torch.uint8, device=DEV)[T % 13:][:stream.size]
        held.copy_(torch.from_numpy(stream))
        out = torch.full((L, T, C), 255, dtype=torch.uint8, device=DEV)
        c_ops.decode_fast_prefsum(held_cdf, held, torch.from_numpy(prefix).to(DEV), out)
        assert np.array_equal(out.cpu().numpy(), want)


# Rows of encode_fast_new: every byte below min(chunk, length) and no other,
# at row strides off the dword, rows that cut their streams, and one to four
# 256-token pieces (a stream's last dword carried from one to the next).
@pytest.mark.parametrize("kind", ["normal", "skewed"])
@pytest.mark.parametrize("L,T,C,nb,chunk", [
    (2, 256, 64, 32, 512), (1, 256, 96, 32, 201), (3, 5, 17, 16, 11), (2, 257, 64, 32, 514), (1, 512, 96, 16, 1024),
    (2, 513, 33, 63, 333), (1, 1000, 64, 32, 1999), (1, 1000, 32, 64, 2), (3, 300, 48, 64, 1),
])
def test_encode_rows_vs_oracle(L, T, C, nb, chunk, kind):
    from lmcache_amd import c_ops

    sym = _symbols(L, T, C, nb, T + C + chunk, kind)
    cdf = oc.calculate_cdf(sym, nb)
    want, want_len = oc.encode(cdf, sym, chunk, out=np.full((L, C, chunk), 0xEE, np.uint8))
    rows = torch.full((L, C, chunk), 0xEE, dtype=torch.uint8, device=DEV)
    lens = torch.full((L, C), -1, dtype=torch.int32, device=DEV)
    c_ops.encode_fast_new(torch.from_numpy(cdf).to(DEV), torch.from_numpy(sym).to(DEV), rows, lens)
    assert np.array_equal(lens.cpu().numpy(), want_len)
    assert np.array_equal(rows.cpu().numpy(), want)


# Streams' places from their lengths (groups of 4096 streams, a last block of
# 32), lengths of another type, and 64-bit sums.
@pytest.mark.parametrize("L,T,C", [(1, 4, 32), (64, 3, 64), (43, 5, 96), (64, 2, 160), (3, 300, 1056)])
def test_decode_chunk_by_lengths(F, L, T, C):
    sym = _symbols(L, T, C, 16, L + T + C)
    chunk = F.encode_chunk(torch.from_numpy(sym).to(DEV), 16)
    other = F.CacheGenChunk(chunk.cdf, chunk.lengths.to(torch.int64), chunk.streams, T)
    assert np.array_equal(F.decode_chunk(chunk).cpu().numpy(), sym)
    assert np.array_equal(F.decode_chunk(other).cpu().numpy(), sym)
    from lmcache_amd import _lib, c_ops

    blocks = (L * C + 63) // 64
    sums = torch.full((blocks + (blocks + 63) // 64,), -1, dtype=torch.int64, device=DEV)
    out = torch.full((L, T, C), 255, dtype=torch.uint8, device=DEV)
    d = [c_ops._desc(t) for t in (chunk.cdf, chunk.streams, chunk.lengths, sums, out)]
    _lib.raise_for(_lib.load().lmc_cachegen_decode(*map(c_ops._ref, d), c_ops._stream(0)))
    assert np.array_equal(out.cpu().numpy(), sym)


# Byte buffers past 2 GiB (64 streams of 40 MB or 64 MiB, their codes in front,
# the last in another group of 4096 streams than most): every decoder takes
# places in 64 bits.
@pytest.mark.parametrize("T", [16, 300, 400, 1025])
@pytest.mark.parametrize("step", [40_000_000, 1 << 26])
def test_decode_chunk_past_2gib(F, T, step):
    L, C = 65, 64
    sym = _symbols(L, T, C, 16, T)
    chunk = F.encode_chunk(torch.from_numpy(sym).to(DEV), 16)
    lens = chunk.lengths.view(-1).tolist()
    wide = list(range(60)) + list(range(L * C - 4, L * C))  # the streams that are spread out
    held = chunk.lengths.view(-1).clone()
    held[wide] = step
    at = np.concatenate([[0], np.cumsum(held.cpu().numpy().astype(np.int64))])
    src = np.concatenate([[0], np.cumsum(np.asarray(lens, np.int64))])
    big = torch.zeros(int(at[-1]), dtype=torch.uint8, device=DEV)
    for s in wide:
        big[at[s]:at[s] + lens[s]] = chunk.streams[src[s]:src[s + 1]]
    big[at[60]:at[L * C - 4]] = chunk.streams[src[60]:src[L * C - 4]]
    assert big.numel() > 2**31
    got = F.decode_chunk(F.CacheGenChunk(chunk.cdf, held.view(L, C), big, T))
    assert np.array_equal(got.cpu().numpy(), sym)


# A stream that reaches almost to 2 GiB.
@pytest.mark.parametrize("T", [16, 300, 400, 1025])
def test_decode_stream_of_almost_2gib(F, T):
    C = 32
    sym = _symbols(1, T, C, 16, T, "constant")
    sym[0, :, 0] = np.arange(T) % 16
    chunk = F.encode_chunk(torch.from_numpy(sym).to(DEV), 16)
    n0, rest = int(chunk.lengths[0, 0]), int(chunk.lengths[0, 1:].sum())
    big = torch.zeros(2**31 - 1, dtype=torch.uint8, device=DEV)
    lens = chunk.lengths.clone()
    for end in (2**31 - 1 - rest, 2**31 - 1):  # with the other streams behind it, or without
        if end == 2**31 - 1:
            lens[0, 1:] = 0
        else:
            big[end:] = chunk.streams[n0:]
        lens[0, 0] = end
        big[:n0] = chunk.streams[:n0]
        got = F.decode_chunk(F.CacheGenChunk(chunk.cdf, lens, big, T)).cpu().numpy()
        assert np.array_equal(got[0, :, 0], sym[0, :, 0])
        if end < 2**31 - 1:
            assert np.array_equal(got, sym)


# Chunks whose quarters do not follow from where they should lie: streams of
# one-bit and of long codes at either end (a quarter outgrows its buffer, or
# starts well off its place), codes of one length (a decoder started between
# boundaries stays between them), the kernel's smallest and largest chunks, and
# chunks below and above that the one-wave decoder takes.
@pytest.mark.parametrize("T", [257, 385, 401, 1000, 1024, 1025])
def test_long_chunk_uneven_streams(F, T):
    L, C, nb = 3, 96, 32
    rng = np.random.default_rng(T)
    sym = np.empty((L, T, C), np.uint8)
    sym[0] = 3
    sym[0, -T // 6:] = rng.integers(0, nb - 1, size=(T // 6 + (T % 6 > 0), C))  # one-bit codes, then five-bit ones
    sym[0, :, 1::2] = sym[0, ::-1, 1::2]
    sym[1] = rng.integers(0, 16, size=(T, C))  # codes of (about) one length
    sym[1, :, :48] = (np.arange(T) % 16)[:, None]  # of exactly one
    sym[2] = _symbols(1, T, C, nb, T)[0]
    sym[2, :, 5] = 7
    chunk = F.encode_chunk(torch.from_numpy(sym).to(DEV), nb)
    assert np.array_equal(F.decode_chunk(chunk).cpu().numpy(), sym)


# The lines between the decoders of long chunks: 384 and 385 tokens, 1024 and
# 1025, and launches of 256 and 257 blocks of 64 streams, with long codes
# (skewed symbols) and short ones.
@pytest.mark.parametrize("kind", ["normal", "skewed"])
@pytest.mark.parametrize("L,T,C", [
    (1, 384, 96), (1, 385, 96), (1, 1024, 96), (1, 1025, 96), (1, 400, 256 * 64), (1, 400, 257 * 64), (257, 401, 64),
])
def test_long_decoder_lines(F, L, T, C, kind):
    sym = np.minimum(_symbols(L, T, C, 32, T + L, kind), 31).astype(np.uint8)
    chunk = F.encode_chunk(torch.from_numpy(sym).to(DEV), 32)
    assert torch.equal(F.decode_chunk(chunk), torch.from_numpy(sym).to(DEV))


# decode_chunk enqueues kernels only, also for the long chunk whose kernel
# takes more than 64 KiB of LDS: captured once, it decodes whatever the chunk's
# buffers hold at each replay.
@pytest.mark.parametrize("T", [200, 300, 1000])
def test_decode_chunk_captured(F, T):
    L, C, nb = 2, 96, 32
    syms = [_symbols(L, T, C, nb, T)]
    rng = np.random.default_rng(T)
    for _ in range(3):  # the same counts per stream: chunks of the same size
        syms.append(np.ascontiguousarray(syms[0][:, rng.permutation(T)]))
    chunks = [F.encode_chunk(torch.from_numpy(s).to(DEV), nb) for s in syms]
    assert len({c.streams.numel() for c in chunks}) == 1
    held = F.CacheGenChunk(chunks[0].cdf.clone(), chunks[0].lengths.clone(), chunks[0].streams.clone(), T)
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        F.decode_chunk(held)
    torch.cuda.current_stream().wait_stream(side)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = F.decode_chunk(held)
    for s, c in zip(syms[1:], chunks[1:]):
        held.cdf.copy_(c.cdf)
        held.lengths.copy_(c.lengths)
        held.streams.copy_(c.streams)
        out.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert np.array_equal(out.cpu().numpy(), s)


def test_encode_chunk_refuses_capture_and_goes_on(F):
    sym = torch.from_numpy(_symbols(2, 40, 64, 16, 5)).to(DEV)
    want = F.encode_chunk(sym, 16)
    side = torch.cuda.Stream()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.stream(side):
        graph.capture_begin()
        try:
            with pytest.raises(RuntimeError, match="cannot be captured"):
                F.encode_chunk(sym, 16)
        finally:
            graph.capture_end()
    torch.cuda.synchronize()
    again = F.encode_chunk(sym, 16)
    assert torch.equal(again.streams, want.streams) and torch.equal(again.cdf, want.cdf)


def test_encode_chunk_from_threads(F):
    """Each thread on its own stream: the words the sizes arrive in are taken
    from one pool."""
    import threading

    syms = [torch.from_numpy(_symbols(2, 100 + 37 * i, 96, 32, i)).to(DEV) for i in range(6)]
    want = [F.encode_chunk(s, 32) for s in syms]
    torch.cuda.synchronize()
    bad = []

    def work(i):
        with torch.cuda.stream(torch.cuda.Stream()):
            for _ in range(20):
                c = F.encode_chunk(syms[i], 32)
                if not torch.equal(c.streams, want[i].streams):
                    bad.append(i)

    threads = [threading.Thread(target=work, args=(i,)) for i in range(len(syms))]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not bad


# The C entries write nothing outside their buffers: each output lies between
# guard bytes, `rows` on a 16-byte boundary and off it, with last blocks of
# one to 33 streams whose bytes end inside a 16-byte vector of their rows.
@pytest.mark.parametrize("shift", [0, 3])
@pytest.mark.parametrize("L,T,C,cap", [
    (1, 1, 1, 2), (1, 3, 5, 6), (3, 7, 33, 14), (1, 2, 3, 4), (1, 3, 2, 6), (1, 7, 1, 14), (2, 1, 33, 2), (5, 3, 13, 6),
    (1, 1, 7, 2), (1, 256, 65, 512), (1, 9, 66, 19), (1, 300, 1, 600), (1, 2, 71, 3),
])
def test_encode_rows_keep_to_their_buffers(L, T, C, cap, shift):
    import ctypes

    from lmcache_amd import _lib, c_ops

    lib, nb, pad = _lib.load(), 16, 256
    sym = _symbols(L, T, C, nb, T + C, "skewed")
    blocks = (L * C + 63) // 64

    def guarded(n, at=pad):
        return torch.full((at + n + pad,), 0xA5, dtype=torch.uint8, device=DEV), at, n

    def part(buf, dtype, shape):
        return buf[0][buf[1]:buf[1] + buf[2]].view(dtype).view(shape)

    cdf = guarded(L * C * (nb + 1) * 2)
    rows = guarded(L * C * cap, pad + shift)
    lens = guarded(L * C * 4)
    off = guarded((2 * blocks + 1) * 8)
    dsym = torch.from_numpy(sym).to(DEV)
    views = [dsym, part(cdf, torch.int16, (L, C, nb + 1)), part(rows, torch.uint8, (L, C, cap)),
             part(lens, torch.int32, (L, C)), part(off, torch.int64, (2 * blocks + 1,))]
    d = [c_ops._desc(v) for v in views]
    total = ctypes.c_int64(-1)
    stream = c_ops._stream(0)
    _lib.raise_for(lib.lmc_cachegen_encode_rows(c_ops._ref(d[0]), nb, *map(c_ops._ref, d[1:]), ctypes.byref(total), stream))
    want_cdf = oc.calculate_cdf(sym, nb)
    want, want_len = oc.encode(want_cdf, sym, cap)
    kept = np.minimum(want_len, cap)
    assert total.value == int(kept.sum())
    streams = guarded(total.value)
    s = c_ops._desc(part(streams, torch.uint8, (total.value,)))
    _lib.raise_for(lib.lmc_cachegen_pack_rows(c_ops._ref(d[2]), c_ops._ref(d[4]), c_ops._ref(s), stream))
    torch.cuda.synchronize()
    for name, (buf, at, n) in dict(cdf=cdf, rows=rows, lens=lens, off=off, streams=streams).items():
        assert bool((buf[:at] == 0xA5).all()) and bool((buf[at + n:] == 0xA5).all()), name
    assert np.array_equal(views[1].cpu().numpy(), want_cdf)
    assert np.array_equal(views[3].cpu().numpy(), want_len)
    got = streams[0][pad:pad + total.value].cpu().numpy()
    assert np.array_equal(got, np.concatenate([want[l, c, :kept[l, c]] for l in range(L) for c in range(C)]))
