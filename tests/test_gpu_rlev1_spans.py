"""RLE v1 columns of few chunks (the launch by spans of all waves) against the
pipelined launch and the oracle: dense and long segments around a step's 8192
bytes, chunks that fill inside a segment, and streams cut, damaged or random."""
import numpy as np
import pytest

import codag_amd as ca
import oracle
from tests import pycodecs as pc
from tests.gpu_helpers import rle_decode, say

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def pair(gpu_required):
    a, b = ca.Context(0), ca.Context(0)
    b.tune_set(ca.RLEV1, ca.TuneParams(512, 2048, 0, 4))  # a chosen shape: the pipeline
    yield a, b
    a.close()
    b.close()


def stream(rng, n, kind):
    s = bytearray()
    while len(s) < n:
        k = kind if kind != "mixed" else rng.choice(["runs", "wide_runs", "ones", "long", "huge"])
        if k == "runs":  # three bytes, all of them terminators
            s += bytes([int(rng.integers(0, 128)), int(rng.integers(0, 128)), int(rng.integers(0, 128))])
        elif k == "wide_runs":  # negative deltas, wide bases
            s += bytes([int(rng.integers(0, 128)), int(rng.integers(128, 256))]) + pc.uleb(int(rng.integers(0, 1 << 62)))
        elif k == "ones":
            s += bytes([255, int(rng.integers(0, 128))])
        elif k == "long":
            s += bytes([128]) + bytes(rng.integers(0, 128, 128, dtype=np.uint8))
        else:
            s += bytes([128]) + b"".join(pc.uleb((1 << 63) + i) for i in range(128))
    return bytes(s)


def compare(contexts, streams, w, chunk):
    off = np.cumsum([0] + [len(s) + i % 17 for i, s in enumerate(streams)]).astype(np.uint64)
    comp = np.zeros(int(off[-1]) + 16, np.uint8)
    for a, s in zip(off, streams):
        comp[int(a):int(a) + len(s)] = np.frombuffer(s, np.uint8)
    cl = np.array([len(s) for s in streams], np.uint64)
    n = len(streams)
    assert n <= 256
    got = [rle_decode(c, ca.RLEV1, comp, off[:-1], cl, w, chunk) for c in contexts]
    ost, oout = oracle.rlev1_decode_chunks(comp, off[:-1], cl, w, chunk, threads=8)
    for st, out in got:
        assert st.tolist() == ost.tolist()
        ok = ost == 0
        assert np.array_equal(out.reshape(n, chunk)[ok], oout.reshape(n, chunk)[ok])
    return ost


@pytest.mark.parametrize("w", [1, 2, 4, 8])
@pytest.mark.parametrize("kind", ["runs", "wide_runs", "ones", "long", "huge", "mixed"])
def test_segments(pair, kind, w):
    say(f"rlev1 spans, {kind}, width {w}")
    rng = np.random.default_rng(60 + w)
    streams = [stream(rng, n, kind) for n in (1, 8180, 8191, 8192, 8193, 16384, 30000)]
    streams += [b"", bytes([0]), bytes([0, 1]), bytes([255])]
    for cap in (1, 63, 64, 65, 4099, 20000):  # chunks that fill within the stream, others that it does not fill
        compare(pair, streams, w, cap * w)


@pytest.mark.parametrize("w", [1, 8])
def test_damaged(pair, w):
    say(f"rlev1 spans, damaged, width {w}")
    rng = np.random.default_rng(70 + w)
    streams = []
    for i in range(60):
        s = bytearray(stream(rng, 12000, "mixed"))
        k = int(rng.integers(0, len(s)))
        if i % 4 == 0:
            s[k:k + int(rng.choice([9, 10, 11, 3000, 9000]))] = b"\xff" * min(9000, len(s) - k)
        elif i % 4 == 1:
            s = s[:k]
        for _ in range(i % 3):
            s[int(rng.integers(0, len(s)))] = int(rng.integers(0, 256))
        streams.append(bytes(s))
    streams += [bytes(rng.integers(0, 256, 9000, dtype=np.uint8)) for _ in range(40)]
    for k in (9, 10, 11, 8170, 9000, 20000):  # overlong varints, with and without an end
        streams += [b"\xff" + b"\x80" * k + b"\x01" + bytes(40), b"\xff" + b"\x80" * k, b"\x05\x81" + b"\x90" * k + b"\x01"]
    # the pipeline reports some varints of over 4 KiB as TRUNCATED
    st = compare(pair[:1], streams, w, 3000 * w)
    assert len(set(st.tolist())) > 2


def test_largest_chunk(pair):
    """2^19 - 1 values a chunk, more than the pipeline's 2^17."""
    say("rlev1 spans, largest chunk")
    rng = np.random.default_rng(80)
    cap = (1 << 19) - 1
    s = bytearray()
    have = 0
    while have < cap:
        n = min(130, cap - have) if cap - have >= 3 else 0
        if n == 0:
            s += bytes([256 - (cap - have)]) + bytes(cap - have)
            have = cap
        else:
            s += bytes([n - 3, int(rng.integers(0, 256))]) + pc.uleb(int(rng.integers(0, 1 << 40)))
            have += n
    st = compare(pair[:1], [bytes(s), bytes(s) + b"\0\0\0", bytes(s[:-4])], 8, cap * 8)
    assert st.tolist() == [0, 0, 1]
