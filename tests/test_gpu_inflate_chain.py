"""Deflate streams whose codes have nearly one length: a decoder that begins at a
wrong bit keeps its wrong phase (7-bit literals read from a bit that is no
multiple of 7), so the span decoder's passes verify a lane or two each and it
goes on with the candidate entries of every lane and a chain through them.
Coded by both group sizes, as batch streams and as chunks, whole and damaged;
every result is compared with zlib's."""
import base64
import zlib

import numpy as np
import pytest

import codag_amd as ca
import oracle
from tests.gpu_helpers import inflate, say
from tests.test_gpu_inflate import Batch, container

pytestmark = pytest.mark.gpu

N = 131072
KINDS = ["symbols128", "symbols64", "base64", "hex"]


def payload(kind, n, seed):
    g = np.random.default_rng(seed)
    if kind.startswith("symbols"):
        return g.integers(0, int(kind[7:]), n, dtype=np.uint8).tobytes()
    if kind == "hex":
        return g.bytes(n // 2 + 1).hex().encode()[:n]
    return base64.b64encode(g.bytes(n))[:n]


def stream(raw, strategy=zlib.Z_HUFFMAN_ONLY, wbits=15):
    c = zlib.compressobj(6, zlib.DEFLATED, wbits, 9, strategy)
    return c.compress(raw) + c.flush()


def coded(kind, strategy=zlib.Z_HUFFMAN_ONLY):
    """Streams of 128 KiB and a remainder, none of them stored."""
    raws = [payload(kind, n, 31 * n + k) for k, n in enumerate((N, N, 65537, 20000, 3001))]
    streams = [stream(r, strategy) for r in raws]
    for s in streams:
        assert (s[2] >> 1) & 3 == 2  # the first block has dynamic codes
    assert all(len(s) < 0.95 * len(r) for s, r in zip(streams, raws))
    return raws, streams


@pytest.fixture(scope="module")
def ctx(gpu_required):
    c = ca.Context(0)
    yield c
    c.close()


@pytest.mark.parametrize("threads", [64, 128])
@pytest.mark.parametrize("kind", KINDS)
def test_batch(ctx, kind, threads):
    say(f"equal code lengths: batch, {kind}, {threads} threads")
    raws, streams = coded(kind)
    more = [stream(r, zlib.Z_DEFAULT_STRATEGY) for r in raws]
    saved = ctx.tune_get(ca.DEFLATE)
    ctx.tune_set(ca.DEFLATE, ca.TuneParams(threads, 0, 12, 1))
    try:
        b = Batch(ctx, streams + more, [len(r) for r in raws * 2])
        for _ in range(2):
            b.launch(0)
            ctx.sync()
        st, written, adler, dst, off = b.results()
    finally:
        ctx.tune_set(ca.DEFLATE, saved)
    for i, r in enumerate(raws * 2):
        assert (st[i], written[i], adler[i]) == (0, len(r), zlib.adler32(r)), i
        assert dst[int(off[i]):int(off[i]) + len(r)].tobytes() == r, i


@pytest.mark.parametrize("waves", [1, 2])  # eight waves a chunk, one wave a chunk
@pytest.mark.parametrize("kind", KINDS)
def test_chunks(ctx, kind, waves):
    """Whole chunks, and chunks cut or damaged after some thousand tokens. The output
    has a spare byte: zlib calls a stream cut in its trailer an overflow where the
    output is full."""
    cap = N + 1
    say(f"equal code lengths: chunks, {kind}, hook {waves}")
    raws, streams = coded(kind)
    rng = np.random.default_rng(len(kind))
    for s in streams[:2]:
        streams.append(s[:len(s) // 2])
        streams.append(s[:len(s) - 3])
        for _ in range(4):
            d = bytearray(s)
            d[int(rng.integers(len(s) // 4, len(s)))] ^= 1 << int(rng.integers(0, 8))
            streams.append(bytes(d))
    comp, off = container(streams)
    try:
        ca.check(ca.lib().codag_test_chunks_two_wave(ctx.h, waves), "test_chunks_two_wave")
        st, ln, out = inflate(ctx, comp, off, cap)
    finally:
        ca.check(ca.lib().codag_test_chunks_two_wave(ctx.h, 0), "test_chunks_two_wave")
    for i in range(len(streams)):
        rc, ref = oracle.zlib_inflate(comp[int(off[i]):int(off[i + 1])].tobytes(), cap)
        assert st[i] == rc, (i, st[i], rc)
        if rc == 0:
            assert ln[i] == len(ref) and out[i * cap:i * cap + len(ref)].tobytes() == ref.tobytes(), i
    assert st[:len(raws)].tolist() == [0] * len(raws)
