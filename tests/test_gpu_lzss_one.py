"""LZSS chunks by the kernel of one wave per chunk with a window, whatever the choice
by the streams would be: KATs, payloads from very compressible to random with chunks
at the edges of its steps (624 stream bytes) and windows (1536 bytes), streams cut and
damaged, chunks that are too small. Everything against the oracle. And the choice."""
import numpy as np
import pytest

import codag_amd as ca
from tests import test_gpu_lzss_parts as lparts
from tests.gpu_helpers import say
from tests.test_gpu_byte_waves import test_lzss_random_and_damaged  # noqa: F401 (runs with this ctx)
from tests.test_gpu_bytecodec import B, LZSS_KATS, compare, lzss_container

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx(gpu_required):
    c = ca.Context(0)
    ca.check(ca.lib().codag_test_byte_waves(c.h, 2), "test_byte_waves")
    yield c
    c.close()


def test_kats(ctx):
    say("lzss by one wave: KATs")
    for s, chunk in LZSS_KATS:
        data, idx = lzss_container([B(s)])
        compare(ctx, True, data, idx, chunk, 3)


@pytest.mark.parametrize("kind", ["noise", "runs", "period", "text"])
@pytest.mark.parametrize("chunk", [1, 17, 554, 555, 1024, 1535, 1536, 1537, 3073, 20000])
def test_whole_and_cut_chunks(ctx, kind, chunk):
    say(f"lzss by one wave: {kind}, chunks of {chunk}")
    raw = lparts.payload(kind, chunk * 3 + chunk // 2)
    data, ends, _, orig = ca.lzss_container(ca.lzss_encode(raw, chunk))
    data, ends = np.array(data), np.array(ends)
    st, ln, out = lparts.decode(ctx, data, ends, chunk, orig)
    assert not st.any() and out[:orig].tobytes() == raw.tobytes() and int(ln.sum()) == orig
    whole = data[:int(ends[0])].tobytes()
    cuts = sorted({min(c, len(whole)) for c in (0, 1, 2, 16, 17, 18, 207, 208, 209, 623, 624, 625, 641, 1247, 1248, 1249,
                                               len(whole) - 1, len(whole))})
    data, idx = lzss_container([whole[:c] for c in cuts])
    for cap in sorted({1, 33, min(chunk, 1536), chunk}):
        compare(ctx, True, data, idx, cap, 7)


def test_choice(ctx):
    say("lzss: the kernel by the streams")
    cus = ctx.info()[1]

    def waves(each, n, chunk):
        return ca.lib().codag_test_lzss_waves(ctx.h, each * n, n, chunk)

    for each, chunk in ((900, 1024), (1153, 1024), (1500, 4096)):
        assert [waves(each, n, chunk) for n in (1, 7 * cus, 7 * cus + 1, 64 * cus)] == [4, 4, 1, 1]
    assert waves(1501, 64 * cus, 4096) == 4 and waves(1400, 64 * cus, 4097) == 4 and waves(1000, 64 * cus, 4097) == 0
    assert [waves(300, 1, c) for c in (1024, 1050, 4096)] == [4, 0, 0] and waves(301, 1, 4096) == 4
    assert waves(0, 1, 1) == 0 and waves(2, 64 * cus, 1) == 1
