"""BRLE and LZSS chunks by each of their kernels, one wave and four waves per chunk,
whatever the choice by the streams would be: KATs, random streams, BRLE streams
whose starts meet soon, late and never, lists, windows and steps at their edges,
LZSS payloads from very compressible to random, streams cut and damaged, chunks
that are too small. Everything against the oracle. And the choice itself, at both
sides of its lines."""
import numpy as np
import pytest

import codag_amd as ca
from tests.gpu_helpers import say
from tests import test_gpu_brle_parts as parts
from tests import test_gpu_lzss_parts as lparts
from tests.test_gpu_bytecodec import (B, BRLE_KATS, LZSS_KATS, brle_container, compare, lzss_container,
                                      random_brle_stream, random_lzss_stream, test_chunks_outside_the_input_are_corrupt)

pytestmark = pytest.mark.gpu
outside = test_chunks_outside_the_input_are_corrupt
del test_chunks_outside_the_input_are_corrupt


@pytest.fixture(scope="module", params=[1, 4])
def ctx(gpu_required, request):
    c = ca.Context(0)
    ca.check(ca.lib().codag_test_byte_waves(c.h, request.param), "test_byte_waves")
    yield c
    c.close()


@pytest.mark.parametrize("lzss", [False, True])
def test_kats(ctx, lzss):
    say(f"byte codecs by waves: KATs, lzss {lzss}")
    for s, chunk in LZSS_KATS if lzss else BRLE_KATS:
        data, idx = (lzss_container if lzss else brle_container)([B(s)])
        compare(ctx, lzss, data, idx, chunk, 3)
    outside(ctx)


def brle_stream(kind, n, rng):
    if kind in ("runs", "high", "ones", "long_runs", "mixed"):
        return parts.stream(kind, n, rng)
    s = bytearray()
    while len(s) < n:
        k = 128 if kind != "any" else int(rng.integers(1, 129))
        if kind == "period":  # the literals repeat, and so do the wrong walks
            r = np.random.default_rng(1)
            s += parts.literal((r.integers(0, 256, 37, dtype=np.uint8).tobytes() * 4)[:k])
        else:
            s += parts.literal(rng.integers(0, 256, k, dtype=np.uint8).tobytes())
        if kind == "change" and len(s) > n // 2:  # from blocks that are passed over to dense ones
            s += parts.stream("mixed", n - len(s), rng)
    return bytes(s)


@pytest.mark.parametrize("kind", ["runs", "high", "ones", "long_runs", "mixed", "noise", "period", "any", "change"])
def test_brle_streams(ctx, kind):
    say(f"brle by waves, {kind}")
    rng = np.random.default_rng(21)
    sizes = [1, 59, 60, 61, 129, 130, 1000, 3839, 3840, 3841, 4100, 7680, 15359, 15360, 15361, 31000]
    streams = [brle_stream(kind, n, rng) for n in sizes]
    data, ptr = brle_container(streams)
    compare(ctx, False, data, ptr, 1 << 20, 5)  # the longest streams of runs overflow
    cut = [s[:max(0, len(s) - int(rng.integers(0, 200)))] for s in streams]
    data, ptr = brle_container(cut)
    for cap in (1, 2047, 2048, 9999, 60000):
        compare(ctx, False, data, ptr, cap, 3)


def test_brle_random_and_damaged(ctx):
    say("brle by waves, random and damaged")
    rng = np.random.default_rng(22)
    streams = []
    for mix in (0.0, 0.2, 0.5, 0.9, 1.0):
        s, _ = random_brle_stream(rng, 50000, mix)
        streams.append(s)
        for _ in range(4):
            d = bytearray(s)
            for _ in range(5):
                d[int(rng.integers(0, len(d)))] = int(rng.integers(0, 256))
            streams.append(bytes(d[:int(rng.integers(1, len(d) + 1))]))
    streams += [rng.integers(0, 256, n, dtype=np.uint8).tobytes() for n in (5, 700, 5000, 40000)] + [b""]
    data, ptr = brle_container(streams)
    for cap in (30000, 65536):
        compare(ctx, False, data, ptr, cap, 7)


@pytest.mark.parametrize("kind", ["noise", "runs", "period", "text"])
def test_lzss_payloads(ctx, kind):
    say(f"lzss by waves, {kind}")
    streams = []
    for n in (1, 17, 1535, 1536, 6145, 50000):
        data, ends, _, _ = ca.lzss_container(ca.lzss_encode(lparts.payload(kind, n), max(n, 1)))
        streams.append(np.array(data)[:int(ends[0])].tobytes())
    streams += [streams[-1][:k] for k in (*range(0, 40), 400, 512, 520, 1000, 1023, 1024, 3119, 3120, 3121) if k < len(streams[-1])]
    data, ends = lzss_container(streams)
    for cap in (1, 100, 4096, 49999, 50000):
        compare(ctx, True, data, ends, cap, 9)


def test_lzss_random_and_damaged(ctx):
    say("lzss by waves, random and damaged")
    rng = np.random.default_rng(23)
    streams = []
    for near in (0.0, 0.3, 0.8, 1.0):
        s, _ = random_lzss_stream(rng, 60000, near)
        streams.append(s)
        for _ in range(5):
            d = bytearray(s)
            for _ in range(3):
                d[int(rng.integers(0, len(d)))] = int(rng.integers(0, 256))
            streams.append(bytes(d[:int(rng.integers(1, len(d) + 1))]))
    streams += [rng.integers(0, 256, n, dtype=np.uint8).tobytes() for n in (5, 700, 5000)] + [b""]
    # matches that repeat 1 to 40 bytes, one after the other
    for d in (1, 2, 3, 7, 33, 34, 35, 40):
        s = bytearray()
        made = 0
        for item in range(4000):
            if item % 8 == 0:
                s.append(0xFF if item < (d + 7) // 8 * 8 else 0)
            if item < (d + 7) // 8 * 8:
                s.append(int(rng.integers(0, 256)))
                made += 1
            else:
                v = (d << 5) | int(rng.integers(0, 32))
                s += bytes([v & 255, v >> 8])
        streams.append(bytes(s))
    data, ends = lzss_container(streams)
    for cap in (30000, 80000):
        compare(ctx, True, data, ends, cap, 11)


def test_choice(ctx):
    say("byte codecs: the choice by the streams")
    cus = ctx.info()[1]

    def one(lzss, each, n, chunk):
        return ca.lib().codag_test_byte_one(ctx.h, lzss, each * n, n, chunk)

    for n in (1, 5 * cus, 100 * cus):
        assert one(0, 4200, n, 262144) == 1
    assert [one(0, 20000, n, 262144) for n in (1, 7 * cus, 7 * cus + 1)] == [0, 0, 1]
    assert [one(0, 100000, n, 262144) for n in (1, 15 * cus, 15 * cus + 1)] == [0, 0, 1]
    assert [one(1, 8000, n, 131072) for n in (1, 2 * cus, 2 * cus + 1)] == [0, 0, 1]
    assert one(1, 100, 1, 1024) == 1 and one(1, 250, 1, 1024) == 1 and one(1, 900, 10 ** 6, 1024) == 0
    assert [one(1, 700, n, 4096) for n in (7 * cus, 7 * cus + 1)] == [0, 1]
    assert [one(1, 20000, n, 131072) for n in (15 * cus, 15 * cus + 1)] == [0, 1]
    assert one(0, 0, 1, 1) == 1 and one(1, 0, 1, 1) == 1
