"""Which kernel an RLE launch takes: the default shape leaves it to the chunk
count, and does so again after it was read, replaced and put back, and after an
autotuner call that failed. The kernels of larger launches (RLE v1: the
pipeline; RLE v2: walker and expanders) give the statuses and values that those
of small launches give, and the oracle's: streams are repeated until there are
more chunks than the small launches take."""
import numpy as np
import pytest

import codag_amd as ca
import oracle
from tests.gpu_helpers import rle_decode, say
from tests import test_gpu_rlev1_spans as v1
from tests import test_gpu_rlev2_spans as v2

pytestmark = pytest.mark.gpu

PC, PIPE, SPAN = 2, 8, 9  # capi.cpp, enum Route


@pytest.fixture(scope="module")
def ctx(gpu_required):
    c = ca.Context(0)
    yield c
    c.close()


def routes(ctx, codec):
    cus = ctx.info()[1]
    return [ca.lib().codag_test_route(ctx.h, codec, n * 30000, n, 4, 131072)
            for n in (1, cus, cus + 1, 2 * cus, 2 * cus + 1, 6 * cus + 1, 12 * cus + 1)]


DEFAULT = {ca.RLEV1: [SPAN, SPAN] + [PIPE] * 5, ca.RLEV2: [SPAN] * 4 + [PC + 3, PC + 2, PC + 1]}


@pytest.mark.parametrize("codec,other,routed", [(ca.RLEV1, (256, 4096, 2), PC + 3), (ca.RLEV2, (192, 4096, 2), PC + 2)])
def test_shape_put_back(ctx, codec, other, routed):
    say(f"rle routes, codec {codec}")
    assert routes(ctx, codec) == DEFAULT[codec]
    saved = ctx.tune_get(codec)
    ctx.tune_set(codec, ctx.tune_get(codec))
    assert routes(ctx, codec) == DEFAULT[codec]
    ctx.tune_set(codec, ca.TuneParams(other[0], other[1], 0, other[2]))
    assert routes(ctx, codec) == [routed] * 7
    ctx.tune_set(codec, saved)
    assert routes(ctx, codec) == DEFAULT[codec]


@pytest.mark.parametrize("codec", [ca.RLEV1, ca.RLEV2])
def test_failed_tune_run_keeps_the_shape(ctx, codec):
    say(f"rle routes after an autotuner call with a bad width, codec {codec}")
    d = ctx.alloc(64)
    with pytest.raises(ca.CodagError):
        ctx.tune_run(codec, d, 8, d, d, 1, 3, 12, d, reps=1)  # 3-byte elements
    assert routes(ctx, codec) == DEFAULT[codec]
    with pytest.raises(ca.CodagError):
        ctx.tune_run(codec, d, 8, d, d, 1 << 60, 1, 16, d, reps=1)  # no room for the statuses
    assert routes(ctx, codec) == DEFAULT[codec]


def repeated(ctx, codec, streams, w, chunk, per_cu):
    """The streams by a small launch, and repeated by one of more than per_cu chunks per CU."""
    n = len(streams)
    off = np.cumsum([0] + [(len(s) + 15) // 16 * 16 + 1 + i % 7 for i, s in enumerate(streams)]).astype(np.uint64)
    comp = np.zeros(int(off[-1]) + 16, np.uint8)
    for a, s in zip(off, streams):
        comp[int(a):int(a) + len(s)] = np.frombuffer(s, np.uint8)
    cl = np.array([len(s) for s in streams], np.uint64)
    k = np.arange(per_cu * ctx.info()[1] + 1) % n
    want = rle_decode(ctx, codec, comp, off[:-1], cl, w, chunk)
    st, out = rle_decode(ctx, codec, comp, off[:-1][k], cl[k], w, chunk)
    assert st.tolist() == want[0][k].tolist()
    out, ref = out.reshape(len(k), chunk), want[1].reshape(n, chunk)
    for i, j in enumerate(k):
        if want[0][j] == 0:
            assert np.array_equal(out[i], ref[j]), (i, j)
    return comp, off, cl, want[0]


@pytest.mark.parametrize("w", [1, 2, 4, 8])
@pytest.mark.parametrize("kind", ["runs", "wide_runs", "ones", "long", "huge", "mixed"])
def test_v1_pipeline_segments(ctx, kind, w):
    say(f"rlev1 pipeline, {kind}, width {w}")
    rng = np.random.default_rng(160 + w)
    streams = [v1.stream(rng, n, kind) for n in (1, 2000, 2048, 8191, 8192, 16384)]
    streams += [b"", bytes([0]), bytes([0, 1]), bytes([255])]
    for cap in (1, 65, 4099, 30000):
        comp, off, cl, st = repeated(ctx, ca.RLEV1, streams, w, cap * w, 1)
        assert st.tolist() == oracle.rlev1_decode_chunks(comp, off[:-1], cl, w, cap * w, threads=8)[0].tolist()


@pytest.mark.parametrize("w", [1, 2, 8])
def test_v1_pipeline_damaged(ctx, w):
    """Damaged streams, overlong varints up to many windows long among them."""
    say(f"rlev1 pipeline, damaged, width {w}")
    rng = np.random.default_rng(170 + w)
    streams = []
    for i in range(40):
        s = bytearray(v1.stream(rng, 9000, "mixed"))
        k = int(rng.integers(0, len(s)))
        if i % 4 == 0:
            s[k:k + int(rng.choice([9, 10, 11, 3000, 9000]))] = b"\xff" * min(9000, len(s) - k)
        elif i % 4 == 1:
            s = s[:k]
        for _ in range(i % 3):
            s[int(rng.integers(0, len(s)))] = int(rng.integers(0, 256))
        streams.append(bytes(s))
    for k in (9, 10, 11, 2040, 4090, 4100, 6000, 8170, 9000, 20000):
        for end in (b"\x01", b"\x01" + bytes(40), b""):
            streams += [b"\xff" + b"\x80" * k + end, b"\x05\x81" + b"\x90" * k + end, b"\x05\x02" + b"\x90" * k + end]
    for cap in (3000, 30000):  # shorter than most streams; room for all
        comp, off, cl, st = repeated(ctx, ca.RLEV1, streams, w, cap * w, 1)
        assert st.tolist() == oracle.rlev1_decode_chunks(comp, off[:-1], cl, w, cap * w, threads=8)[0].tolist()
        assert {1, 3} <= set(st.tolist())


@pytest.mark.parametrize("w", [1, 2, 4, 8])
def test_v2_walker_blocks(ctx, w):
    say(f"rlev2 walker and expanders, width {w}")
    rng = np.random.default_rng(180 + w)
    streams = v2.streams_of(rng, 9000, 24) + [b"", b"\x00", b"\x01\x02"]
    for i in range(24):
        s = bytearray(streams[i])
        for _ in range(1 + i % 3):
            s[int(rng.integers(0, len(s)))] = int(rng.integers(0, 256))
        streams.append(bytes(s[:len(s) if i % 2 else int(rng.integers(1, len(s)))]))
    for cap in (700, 60000):
        repeated(ctx, ca.RLEV2, streams, w, cap * w, 2)


def test_v2_routes_by_bytes(ctx):
    """Streams of up to 128 bytes, and from 3.5 (2.25 above one chunk per CU) stream bytes a value on."""
    say("rlev2 routes by bytes")
    cus = ctx.info()[1]

    def route(comp_bytes, n):
        return ca.lib().codag_test_route(ctx.h, ca.RLEV2, comp_bytes, n, 8, 8192)  # 1024 values a chunk

    for n in (1, cus, cus + 1, 2 * cus):
        line = n * (3584 if n <= cus else 2304)
        assert route(128 * n + 1, n) == SPAN and route(128 * n, n) == PC + 1
        assert route(line, n) == SPAN and route(line + 16, n) == PC + 1
    assert route(2304 * 3 * cus, 3 * cus) == PC + 3 and route(2304 * 3 * cus + 16, 3 * cus) == PC + 1
    assert route((1 << 64) - 1, 2 * cus) == PC + 1 and route(0, 1) == PC + 1


def test_v1_routes_by_bytes(ctx):
    say("rlev1 routes by bytes")
    for w, above in ((1, PIPE), (2, PIPE), (4, SPAN), (8, SPAN)):
        for n in (1, ctx.info()[1]):
            line = n * 8192 * 5 // 4
            got = [ca.lib().codag_test_route(ctx.h, ca.RLEV1, b, n, w, 8192) for b in (line, line + 5)]
            assert got == [SPAN, above]


def test_v1_random_narrow_columns(ctx):
    """Columns at both sides of that line, by one launch each."""
    say("rlev1 random narrow columns")
    rng = np.random.default_rng(9)
    for w, top in ((1, 100), (1, 256), (2, 16000), (2, 65536)):
        raw = rng.integers(0, top, 20 * 4096 // w).astype("u%d" % w)
        cont, off, ln, nc = ca.rlev1_encode(raw, w, 4096)
        n = 20  # the container's last chunks are padding
        st, out = rle_decode(ctx, ca.RLEV1, cont[8:8 + int(off[n - 1] + ln[n - 1])], off[:n], ln[:n], w, 4096)
        assert not st.any() and out.tobytes() == raw.tobytes()


@pytest.mark.parametrize("bits,w", [(64, 8), (40, 8), (32, 4), (20, 4), (0, 8)])
def test_v2_wide_and_tiny_columns(ctx, bits, w):
    """Random values of so many bits, or equal ones, around the chunk counts where the kernel changes."""
    say(f"rlev2 wide columns, {bits} bits, width {w}")
    rng = np.random.default_rng(bits + w)
    cus, chunk = ctx.info()[1], 2048
    m = (2 * cus + 1) * (chunk // w)
    raw = (rng.integers(0, 1 << 63, m, dtype=np.uint64) << np.uint64(1) >> np.uint64(64 - bits) if bits else
           np.full(m, 5)).astype("u%d" % w)
    comp, off, ln, nc = ca.rlev2_encode(raw, w, chunk)
    for n in (1, cus, cus + 1, 2 * cus, 2 * cus + 1):
        st, out = rle_decode(ctx, ca.RLEV2, comp[:int(off[n - 1] + ln[n - 1])], off[:n], ln[:n], w, chunk)
        assert not st.any() and out.tobytes() == raw[:n * (chunk // w)].tobytes()
