"""BRLE chunks at the edges of the decoder's steps (15360 stream bytes in blocks
of 60), lists (512 items) and output windows (2048 bytes), against the oracle:
streams in which a walk from a wrong byte never meets the right one, items of
one size throughout, and steps that end inside an item or at the chunk's end."""
import numpy as np
import pytest

import codag_amd as ca
from tests.gpu_helpers import say
from tests.test_gpu_bytecodec import brle_container, compare

pytestmark = pytest.mark.gpu
STEP = 256 * 60


@pytest.fixture(scope="module")
def ctx(gpu_required):
    c = ca.Context(0)
    yield c
    c.close()


def literal(data):
    return bytes([127 + len(data)]) + bytes(data)


def stream(kind, n, rng):
    """About n stream bytes of items."""
    s = bytearray()
    while len(s) < n:
        if kind == "runs":  # values below 128: every byte could be a header
            s += bytes(rng.integers(0, 128, 2, dtype=np.uint8))
            if rng.integers(0, 400) == 0:  # changes the parity
                s += literal(b"ab")
        elif kind == "high":  # literals whose bytes jump as far as their own header
            s += literal(bytes([255, 254] * 64))
        elif kind == "ones":
            s += literal(bytes(rng.integers(0, 256, 1, dtype=np.uint8)))
        elif kind == "long_runs":
            s += bytes([127, int(rng.integers(0, 256))])
        else:
            k = int(rng.choice([1, 2, 3, 4, 5, 7, 64, 127, 128]))
            s += literal(bytes(rng.integers(0, 256, k, dtype=np.uint8)))
            s += bytes([int(rng.choice([0, 1, 2, 60, 127])), int(rng.integers(0, 256))])
    return bytes(s)


@pytest.mark.parametrize("shift", [0, 5])
@pytest.mark.parametrize("kind", ["runs", "high", "ones", "long_runs", "mixed"])
def test_streams(ctx, kind, shift):
    say(f"brle parts, {kind}, shift {shift}")
    rng = np.random.default_rng(5)
    sizes = [1, 59, 60, 61, 3840, STEP - 1, STEP, STEP + 1, 2 * STEP + 77]
    data, ptr = brle_container([stream(kind, n, rng) for n in sizes])
    compare(ctx, False, data, ptr, 1 << 20, shift)  # the longest streams of runs overflow


@pytest.mark.parametrize("cut", [-130, -2, -1, 0, 1, 2])
def test_stops(ctx, cut):
    """Streams that end, and chunks that fill, around the end of a step."""
    say(f"brle parts, stops {cut}")
    rng = np.random.default_rng(6)
    for kind in ("mixed", "high", "runs"):
        full = stream(kind, 2 * STEP, rng)
        data, ptr = brle_container([full[: STEP + cut], full[: 2 * STEP + cut - 40], full])
        compare(ctx, False, data, ptr, 1 << 20)
        for cap in (1, 2047 + cut, 2048 + cut % 16, 40000 + cut):
            compare(ctx, False, data, ptr, cap, 3)
