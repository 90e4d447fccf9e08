"""RLE v2 columns of few chunks (the launch by spans of all waves) against the
launch by one walker and expanders: the same outputs and statuses on encoder
columns, on blocks of every size around a step's 4096 positions, and on streams
cut, damaged or random."""
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
    b.tune_set(ca.RLEV2, ca.TuneParams(128, 4096, 0, 2))  # a chosen shape: the walker
    yield a, b
    a.close()
    b.close()


def streams_of(rng, n, count):
    """Streams of about n bytes of blocks of every kind."""
    out = []
    for _ in range(count):
        s = bytearray()
        while len(s) < n:
            kind = rng.integers(0, 6)
            if kind <= 1:
                s += pc.v2_short_repeat(int(rng.integers(0, 1 << 16)), int(rng.integers(3, 11)), int(rng.integers(2, 9)))
            elif kind == 2:
                code = int(rng.integers(0, 32))
                bits = min(pc.DECODE_WIDTHS[code], 62)
                s += pc.v2_direct([int(x) for x in rng.integers(0, 1 << bits, int(rng.choice([1, 5, 64, 128, 255])))], code)
            elif kind == 3:
                s += pc.v2_delta(int(rng.integers(0, 1 << 62)), int(rng.integers(-9, 9)),
                                 [int(x) for x in rng.integers(0, 128, int(rng.integers(1, 200)))], 7)
            elif kind == 4:
                s += pc.v2_delta(5, int(rng.integers(-3, 4)), [0] * int(rng.integers(1, 100)), None)
            else:
                red = [int(x) for x in rng.integers(0, 8, 128)]
                s += pc.v2_patched_base(red, 1000, 2, 2, [(70, 5), (57, 9)], 3, 8)
        out.append(bytes(s))
    return out


def compare(pair, streams, w, chunk):
    off = np.cumsum([0] + [(len(s) + 15) // 16 * 16 + 1 for s in streams]).astype(np.uint64)  # odd begins
    comp = np.zeros(int(off[-1]) + 16, np.uint8)
    for a, s in zip(off, streams):
        comp[int(a):int(a) + len(s)] = np.frombuffer(s, np.uint8)
    cl = np.array([len(s) for s in streams], np.uint64)
    got = [rle_decode(c, ca.RLEV2, comp, off[:-1], cl, w, chunk) for c in pair]
    assert got[0][0].tolist() == got[1][0].tolist()
    ok = got[0][0] == 0
    n = len(streams)
    assert np.array_equal(got[0][1].reshape(n, chunk)[ok], got[1][1].reshape(n, chunk)[ok])
    for i in np.flatnonzero(ok)[:4]:  # and the oracle's
        rc, ref = oracle.rlev2_decode_chunk(streams[i], w, chunk // w)
        assert rc == 0 and np.array_equal(got[0][1].reshape(n, chunk)[i].view(ref.dtype)[:len(ref)], ref)
    return got[0][0]


@pytest.mark.parametrize("w", [1, 2, 4, 8])
def test_blocks(pair, w):
    say(f"rlev2 spans, blocks, width {w}")
    rng = np.random.default_rng(40 + w)
    streams = [x for n in (1, 60, 4000, 4096, 4200, 8192, 20000) for x in streams_of(rng, n, 6)]
    st = compare(pair, streams, w, (1 << 18) - 64)
    assert (st == 0).any()
    compare(pair, streams, w, 5000 * w)  # the longer ones overflow


def test_dense_and_largest_blocks(pair):
    """2048 blocks a step, and blocks of 2042 bytes across its end."""
    say("rlev2 spans, dense and largest")
    big = pc.v2_direct([(1 << 61) + i for i in range(255)], 31)
    streams = [bytes([0x00, 7]) * 9000, big * 9, bytes([0x00, 7]) * 2047 + big * 2, bytes([0x00, 7]) * 2048 + big,
               b"", bytes([0x00])]
    compare(pair, streams, 8, 1 << 19)


@pytest.mark.parametrize("w", [2, 8])
def test_damaged(pair, w):
    say(f"rlev2 spans, damaged, width {w}")
    rng = np.random.default_rng(50 + w)
    streams = []
    for s in streams_of(rng, 9000, 40):
        streams.append(s[: int(rng.integers(0, len(s)))])
        t = bytearray(s)
        for _ in range(3):
            t[int(rng.integers(0, len(t)))] = int(rng.integers(0, 256))
        streams.append(bytes(t))
    streams += [bytes(rng.integers(0, 256, 6000, dtype=np.uint8)) for _ in range(40)]
    # varints of 10 and more bytes, and ones that the step's search does not reach
    for k in (9, 10, 11, 70, 5000):
        streams.append(bytes([0x00, 7]) * 30 + bytes([0xC0, 0x02]) + b"\x80" * k + b"\x01\x02" + bytes([0x00, 7]) * 9)
    compare(pair, streams, w, (1 << 18) - 64)
