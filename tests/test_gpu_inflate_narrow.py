"""Very compressible Deflate streams, which are decoded 64 bits at a time with
their matches copied one after the other through a ring of the last output bytes:
distances around a lane row, a match and the ring's size, repeats shorter than
their match, sources in and before the ring, changes from compressible to plain
bytes and back, outputs that are exact, roomy and too small, streams cut and
damaged; by both group sizes. Whole streams give zlib's bytes and check values,
the others zlib's status, and the same bytes by both group sizes."""
import zlib

import numpy as np
import pytest

import codag_amd as ca
import oracle
from tests.gpu_helpers import inflate, say
from tests.test_gpu_inflate import container

pytestmark = pytest.mark.gpu

DTYPE = np.dtype([("bytes", "<u8"), ("status", "<i4"), ("adler", "<u4")])


@pytest.fixture(scope="module")
def ctx(gpu_required):
    c = ca.Context(0)
    yield c
    c.close()


def z(raw, level=9, strategy=zlib.Z_DEFAULT_STRATEGY, wbits=15):
    c = zlib.compressobj(level, zlib.DEFLATED, wbits, 9, strategy)
    return c.compress(raw) + c.flush()


def noise(n, seed):
    return np.random.default_rng(seed).integers(0, 256, n, dtype=np.uint8).tobytes()


def sparse(n, gap, seed):
    return (np.random.default_rng(seed).integers(0, gap, n) == 0).astype(np.uint8).tobytes()


def payloads():
    out = {"zeros%d" % n: bytes(n) for n in (1, 257, 258, 259, 1023, 1024, 1025, 2047, 2048, 2049, 8191, 8193, 32769, 70001, 1 << 20)}
    for d in (1, 2, 3, 4, 5, 63, 64, 65, 127, 129, 255, 256, 257, 258, 259, 300, 1000, 4000, 6143, 6144, 6145, 8192, 20000, 30719, 30720, 32768):
        n = max(60 * d, 60000) if d < 1000 else 9 * d + 7
        out["period%d" % d] = (noise(d, d) * (n // d + 1))[:n]
    out["sparse"] = sparse(300000, 200, 1)
    out["sparse2k"] = sparse(400000, 2000, 2)
    text = ca.synth_deflate_payload(50000, 5000, seed=5).tobytes()
    out["mixed"] = bytes(90000) + text + b"abcde" * 20000 + noise(3000, 3) + bytes(70000) + text[:9999] + sparse(200000, 900, 4)
    return out


def run(ctx, streams, caps, threads, flags=0):
    """Status, bytes, check value and output of each stream, source and output at odd places."""
    src, at, to, n = bytearray(), [], [], 0
    for k, (s, c) in enumerate(zip(streams, caps)):
        src += bytes(k % 5)
        at.append(len(src))
        src += s
        to.append(n + k % 7)
        n = to[-1] + c + 1
    d_src, d_dst = ctx.upload(np.frombuffer(bytes(src) + bytes(16), np.uint8)), ctx.alloc(n + 16)
    d_dst.fill(0xA5)
    d = np.zeros((len(streams), 4), np.uint64)
    d[:, 0] = d_src.ptr.value + np.array(at, np.uint64)
    d[:, 1] = [len(s) for s in streams]
    d[:, 2] = d_dst.ptr.value + np.array(to, np.uint64)
    d[:, 3] = caps
    d_descs, d_res = ctx.upload(d), ctx.alloc(16 * len(streams))
    saved = ctx.tune_get(ca.DEFLATE)
    ctx.tune_set(ca.DEFLATE, ca.TuneParams(threads, 0, 12, 1))
    try:
        ctx.inflate_batch(d_descs, len(streams), d_res, flags)
        ctx.sync()
    finally:
        ctx.tune_set(ca.DEFLATE, saved)
    res, out = d_res.download().view(DTYPE), d_dst.download()
    return res, [out[a:a + c + 1] for a, c in zip(to, caps)]


@pytest.mark.parametrize("threads", [64, 128])
def test_whole(ctx, threads):
    say(f"compressible streams, {threads} threads")
    p = payloads()
    raws, streams, caps = [], [], []
    for raw in p.values():
        for s in (z(raw), z(raw, 6, zlib.Z_FIXED)):
            for cap in (len(raw), 3 * len(raw) + 100):
                raws.append(raw)
                streams.append(s)
                caps.append(cap)
    # a plain text with room for 1000 times its bytes
    text = ca.synth_deflate_payload(20000, 5000, seed=8).tobytes()
    raws.append(text)
    streams.append(z(text))
    caps.append(1000 * len(streams[-1]))
    res, out = run(ctx, streams, caps, threads)
    for i, r in enumerate(raws):
        assert (res["status"][i], res["bytes"][i], res["adler"][i]) == (0, len(r), zlib.adler32(r)), i
        assert out[i][:len(r)].tobytes() == r and (out[i][len(r):] == 0xA5).all(), i


@pytest.mark.parametrize("threads", [64, 128])
def test_gzip_and_raw(ctx, threads):
    say(f"compressible gzip and raw streams, {threads} threads")
    raws = [r for k, r in payloads().items() if k in ("zeros70001", "period37", "period300", "sparse", "mixed", "period5")]
    for wbits, flags, check in ((31, ca.INFLATE_GZIP, zlib.crc32), (-15, ca.INFLATE_RAW, zlib.adler32)):
        res, out = run(ctx, [z(r, 9, wbits=wbits) for r in raws], [len(r) for r in raws], threads, flags)
        for i, r in enumerate(raws):
            assert (res["status"][i], res["bytes"][i], res["adler"][i]) == (0, len(r), check(r)), i
            assert out[i][:len(r)].tobytes() == r, i


def test_cut_damaged_and_too_small(ctx):
    say("compressible streams, cut, damaged, too small outputs")
    rng = np.random.default_rng(11)
    streams, caps = [], []
    for name in ("zeros70001", "period3", "period64", "period300", "sparse", "sparse2k", "mixed", "period8192"):
        raw = payloads()[name]
        s = z(raw)
        for cap in (0, 1, 257, 1000, 2048, 5000, len(raw) // 2, len(raw) - 1):
            streams.append(s)
            caps.append(cap)
        for k in rng.integers(1, len(s), 12):
            streams.append(s[:int(k)])
            caps.append(len(raw) + 1)
        for _ in range(24):
            d = bytearray(s)
            d[int(rng.integers(2, len(s)))] ^= 1 << int(rng.integers(0, 8))
            streams.append(bytes(d))
            caps.append(len(raw) + 4000)
    one, out1 = run(ctx, streams, caps, 64)
    many, out8 = run(ctx, streams, caps, 128)
    assert one.tolist() == many.tolist()
    seen = set()
    for i, (s, c) in enumerate(zip(streams, caps)):
        n = int(one["bytes"][i])
        assert n <= c and np.array_equal(out1[i][:n], out8[i][:n]), i
        assert out1[i][c] == 0xA5 and out8[i][c] == 0xA5, i
        rc, ref = oracle.zlib_inflate(s, c)
        # where a match both passes the output's end and reaches too far back, zlib, which
        # writes what fits, names the distance
        assert one["status"][i] == rc or (one["status"][i], rc) == (2, 3), (i, one["status"][i], rc)
        if rc == 0:
            assert out1[i][:n].tobytes() == ref.tobytes(), i
        seen.add(rc)
    assert {1, 2, 3} <= seen


@pytest.mark.parametrize("waves", [1, 2])
def test_chunks(ctx, waves):
    say(f"compressible chunks, hook {waves}")
    cap = 65536 + 13
    raws = [r[:cap] for r in payloads().values()]
    streams = [z(r, 6) for r in raws]
    comp, off = container(streams)
    try:
        ca.check(ca.lib().codag_test_chunks_two_wave(ctx.h, waves), "test_chunks_two_wave")
        st, ln, out = inflate(ctx, comp, off, cap)
    finally:
        ca.check(ca.lib().codag_test_chunks_two_wave(ctx.h, 0), "test_chunks_two_wave")
    for i, r in enumerate(raws):
        assert (st[i], ln[i]) == (0, len(r)) and out[i * cap:i * cap + len(r)].tobytes() == r, i
