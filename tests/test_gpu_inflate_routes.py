"""How many waves decode a Deflate chunk: by the chunk count, the chunk's size and
the streams' bytes. The rule at both sides of its lines, and containers decoded
there."""
import numpy as np
import pytest

import codag_amd as ca
from tests.gpu_helpers import inflate, say

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx(gpu_required):
    c = ca.Context(0)
    yield c
    c.close()


def many(ctx, n, chunk, ratio):
    return ca.lib().codag_test_inflate_many(ctx.h, int(n * chunk * ratio), n, chunk)


def test_lines(ctx):
    say("inflate routes")
    cus = ctx.info()[1]
    for n in (1, cus, 2 * cus):
        for ratio in (0.001, 0.5, 0.8, 1.0, 5.0):
            assert many(ctx, n, 131072, ratio) and many(ctx, n, 4097, ratio)
        assert [many(ctx, n, 4096, r) for r in (0.05, 0.13, 0.5, 0.64, 0.7, 1.0)] == [0, 1, 1, 1, 0, 0]
    for n in (2 * cus + 1, 5 * cus):
        for chunk in (8193, 131072):
            assert [many(ctx, n, chunk, r) for r in (0.001, 0.03, 0.04, 0.5, 0.64, 0.7, 0.98, 1.0)] == [0, 0, 1, 1, 1, 0, 0, 1]
        assert not any(many(ctx, n, chunk, r) for chunk in (1, 256, 8192) for r in (0.01, 0.5, 1.0))
    for n in (5 * cus + 1, 1 << 20):
        assert not any(many(ctx, n, 131072, r) for r in (0.01, 0.5, 1.0))
    assert ca.lib().codag_test_inflate_many(ctx.h, 0, 1, 131072) == 1


@pytest.mark.parametrize("kind", ["text", "zeros", "letters", "noise"])
def test_containers(ctx, kind):
    """Around two and five chunks per CU, of 2000 and 9000 bytes."""
    say(f"inflate containers, {kind}")
    cus = ctx.info()[1]
    rng = np.random.default_rng(len(kind))
    for chunk in (2000, 9000):
        total = (5 * cus + 1) * chunk
        raw = {"text": lambda: ca.synth_deflate_payload(total, chunk, seed=3),
               "zeros": lambda: np.zeros(total, np.uint8),
               "letters": lambda: rng.integers(0, 100, total, dtype=np.uint8),
               "noise": lambda: rng.integers(0, 256, total, dtype=np.uint8)}[kind]()
        comp, blk, _, nc = ca.deflate_compress_chunks(raw, chunk, level=6)
        off = blk[1:]
        for n in (2 * cus, 2 * cus + 1, 5 * cus, 5 * cus + 1):
            st, ln, out = inflate(ctx, comp[:int(off[n])], off[:n + 1], chunk)
            assert not st.any() and (ln == chunk).all() and out.tobytes() == raw[:n * chunk].tobytes()
