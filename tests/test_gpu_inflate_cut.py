"""Deflate streams that end early: cut after every byte, block headers and codes
included, with the bytes behind the cut still lying in memory (an error that
only those bits would make is none yet), and random block headers. Statuses are
zlib's, by both group sizes."""
import zlib

import numpy as np
import pytest

import codag_amd as ca
import oracle
from tests.gpu_helpers import say

pytestmark = pytest.mark.gpu


class Bits:
    """A raw Deflate stream bit by bit."""

    def __init__(self):
        self.v, self.n = 0, 0

    def put(self, value, n):  # least significant bit first
        self.v |= value << self.n
        self.n += n
        return self

    def code(self, value, n):  # a Huffman code, most significant bit first
        return self.put(int(format(value, "0%db" % n)[::-1], 2), n)

    def bytes(self):
        return self.v.to_bytes((self.n + 7) // 8, "little")


def header(nlen, ndist, code_lens):
    """A dynamic block up to its code lengths; code_lens by position in the stream."""
    b = Bits().put(1, 1).put(2, 2).put(nlen - 257, 5).put(ndist - 1, 5).put(len(code_lens) - 4, 4)
    for x in code_lens:
        b.put(x, 3)
    return b


def crafted():
    """Raw streams with an error at a known place, some bytes behind it."""
    tail = bytes(range(1, 90))
    out = []
    # the code-length codes over-subscribed, incomplete, and none at all
    out += [header(257, 1, [1] * 19).bytes() + tail, header(257, 1, [7] * 19).bytes() + tail,
            header(286, 30, [0] * 19).bytes() + tail, header(287, 30, [1, 1, 0, 0]).bytes() + tail]
    # a repeat of the last length at the front; one that runs past the end
    out.append(header(257, 1, [1, 0, 0, 1]).code(1, 1).put(3, 2).bytes() + tail)
    b = header(257, 1, [0, 0, 1, 1])  # 18 -> code 1, 0 -> code 0
    for _ in range(2):
        b.code(1, 1).put(127, 7)
    out.append(b.bytes() + tail)
    # fixed codes: length codes 286 and 287, distance codes 30 and 31
    for sym in (198, 199):
        out.append(Bits().put(1, 1).put(1, 2).code(0x30, 8).code(sym, 8).bytes() + tail)
    for d in (30, 31):
        b = Bits().put(1, 1).put(1, 2)
        for _ in range(5):
            b.code(0x41, 8)
        out.append(b.code(1, 7).code(d, 5).bytes() + tail)
    return out


def cuts():
    text = ca.synth_deflate_payload(6000, 3000, seed=4).tobytes()
    g = np.random.default_rng(6)
    whole = []
    for level, strategy in ((6, 0), (9, 0), (6, zlib.Z_HUFFMAN_ONLY), (6, zlib.Z_RLE), (6, zlib.Z_FIXED)):
        for raw in (text[:700], g.integers(0, 40, 300, dtype=np.uint8).tobytes(), b"ab" * 400):
            c = zlib.compressobj(level, zlib.DEFLATED, -15, 8, strategy)
            whole.append(c.compress(raw) + c.flush())
    whole += crafted()
    return [(s, k) for s in whole for k in range(min(len(s), 260) + 1)]


def garbage():
    g = np.random.default_rng(7)
    out = []
    for i in range(3000):
        s = bytearray(g.bytes(int(g.integers(8, 120))))
        s[0] = (s[0] & ~7) | 1 | (2 if i % 4 == 0 else 4)  # the last block, mostly dynamic
        if i % 2:
            s[1] &= 0xf0  # few length codes
        out.append((bytes(s), int(g.integers(0, len(s) + 1))))
    return out


def decode(ctx, streams, cap, threads):
    """Statuses of the raw streams' first k bytes; the bytes behind lie there too."""
    at = np.cumsum([0] + [len(s) for s, _ in streams])
    src = ctx.upload(np.frombuffer(b"".join(s for s, _ in streams) + bytes(16), np.uint8))
    n = len(streams)
    dst, res = ctx.alloc(n * cap), ctx.alloc(16 * n)
    d = np.zeros((n, 4), np.uint64)
    d[:, 0] = src.ptr.value + at[:-1].astype(np.uint64)
    d[:, 1] = [k for _, k in streams]
    d[:, 2] = dst.ptr.value + np.arange(n, dtype=np.uint64) * np.uint64(cap)
    d[:, 3] = cap
    descs = ctx.upload(d)
    saved = ctx.tune_get(ca.DEFLATE)
    ctx.tune_set(ca.DEFLATE, ca.TuneParams(threads, 0, 12, 1))
    try:
        ctx.inflate_batch(descs, n, res, ca.INFLATE_RAW)
        ctx.sync()
    finally:
        ctx.tune_set(ca.DEFLATE, saved)
    return res.download(16 * n).view(np.int32).reshape(n, 4)[:, 2]


@pytest.mark.parametrize("threads", [64, 128])
@pytest.mark.parametrize("which", ["cuts", "garbage"])
def test_statuses(which, threads):
    say(f"inflate, streams that end early: {which}, {threads} threads")
    streams = cuts() if which == "cuts" else garbage()
    cap = 40000 if which == "garbage" else 2000
    seen = set()
    with ca.Context(0) as ctx:
        step = 400  # at most two streams per CU: eight-wave groups with 128 threads
        for a in range(0, len(streams), step):
            part = streams[a:a + step]
            st = decode(ctx, part, cap, threads)
            for i, (s, k) in enumerate(part):
                rc, _ = oracle.zlib_inflate(s[:k], cap, raw=True)
                assert st[i] == rc, (a + i, k, len(s), s[:12].hex(), st[i], rc)
                seen.add(rc)
    assert {1, 3} <= seen
