"""Edges of the Deflate span decoder: outputs around its window and segment
sizes, codes of every length, tokens that never stop, streams that do not
synchronise, and the counts at which the launches change their shape. Every
output is compared with zlib's input; statuses and check values must hold."""
import zlib

import numpy as np
import pytest

import codag_amd as ca
from tests.gpu_helpers import say

pytestmark = pytest.mark.gpu

DTYPE = np.dtype([("bytes", "<u8"), ("status", "<i4"), ("adler", "<u4")])


def payload(kind, n):
    g = np.random.default_rng(n * 7 + len(kind))
    if kind == "noise":  # literals of about eight bits each
        return g.integers(0, 256, n, dtype=np.uint8).tobytes()
    if kind == "runs":  # matches of 258 bytes at distance 1
        return bytes(n)
    if kind == "period":  # overlapping matches at a short distance
        return (g.integers(0, 256, 37, dtype=np.uint8).tobytes() * (n // 37 + 1))[:n]
    if kind == "skewed":  # code lengths up to 15 bits
        fib = [1, 1]
        while len(fib) < 24:
            fib.append(fib[-1] + fib[-2])
        p = np.array(fib, np.float64)
        return g.choice(24, n, p=p / p.sum()).astype(np.uint8).tobytes()
    if kind == "two":  # one-bit codes
        return (g.integers(0, 40, n) == 0).astype(np.uint8).tobytes()
    return ca.synth_deflate_payload(max(n, 1), 5000, seed=n)[:n].tobytes()


def stream(raw, strategy=zlib.Z_DEFAULT_STRATEGY, level=6):
    c = zlib.compressobj(level, zlib.DEFLATED, 15, 9, strategy)
    return c.compress(raw) + c.flush()


def run_batch(ctx, raws, streams, threads):
    """Each stream at its own alignment, each output with one byte to spare."""
    src, at = bytearray(), []
    for k, s in enumerate(streams):
        src += bytes(k % 5)
        at.append(len(src))
        src += s
    d_src = ctx.upload(np.frombuffer(bytes(src) + bytes(16), np.uint8))
    off = np.concatenate([[0], np.cumsum([len(r) + 1 for r in raws])])
    d_dst = ctx.alloc(int(off[-1]) + 16)
    d_dst.fill(0xA5)
    d = np.zeros((len(raws), 4), np.uint64)
    d[:, 0] = d_src.ptr.value + np.array(at, np.uint64)
    d[:, 1] = [len(s) for s in streams]
    d[:, 2] = d_dst.ptr.value + off[:-1].astype(np.uint64)
    d[:, 3] = [len(r) for r in raws]
    d_descs, d_res = ctx.upload(d), ctx.alloc(16 * len(raws))
    ctx.tune_set(ca.DEFLATE, ca.TuneParams(threads, 0, 12, 1))
    ctx.inflate_batch(d_descs, len(raws), d_res)
    ctx.sync()
    res, out = d_res.download().view(DTYPE), d_dst.download()
    for k, r in enumerate(raws):
        assert (res["status"][k], res["bytes"][k], res["adler"][k]) == (0, len(r), zlib.adler32(r)), k
        assert out[off[k]:off[k + 1] - 1].tobytes() == r, k
        assert out[off[k + 1] - 1] == 0xA5, k


@pytest.mark.parametrize("threads", [64, 128])
@pytest.mark.parametrize("kind", ["noise", "runs", "period", "skewed", "two", "mixed"])
def test_window_and_segment_edges(kind, threads):
    say(f"span decoder: {kind}, {threads} threads")
    sizes = [1, 2, 63, 64, 65, 255, 257, 2559, 2560, 2561, 4095, 4096, 4097, 5120, 8192, 20479, 20480, 20481, 65537, 150001]
    raws = [payload(kind, n) for n in sizes for _ in range(3)]
    strategies = [zlib.Z_DEFAULT_STRATEGY, zlib.Z_HUFFMAN_ONLY, zlib.Z_FIXED]
    streams = [stream(r, strategies[i % 3]) for i, r in enumerate(raws)]
    with ca.Context(0) as ctx:
        run_batch(ctx, raws, streams, threads)


@pytest.mark.parametrize("sizes", ["small", "uneven"])
@pytest.mark.parametrize("over", [0, 1])
def test_batch_shapes_by_size(sizes, over):
    """At two streams per CU and one more, and far above, where the plan picks
    one wave per stream for small streams and eight for uneven ones."""
    with ca.Context(0) as ctx:
        cus = ctx.info()[1]
        say(f"batch plan: {sizes}, {cus} CUs")
        n = 2 * cus + over if over == 0 or sizes == "uneven" else 16 * cus + 1
        raws = [payload("mixed", 300 + k % 700) for k in range(n)]
        if sizes == "uneven":
            raws[0] = payload("mixed", 1 << 20)
        run_batch(ctx, raws, [stream(r) for r in raws], 128)


@pytest.mark.parametrize("per_cu,chunk", [(5, 1000), (6, 1000), (1, 70000)])
def test_chunk_counts(per_cu, chunk):
    with ca.Context(0) as ctx:
        n = ctx.info()[1] * per_cu
        say(f"chunk container: {n} chunks of {chunk} bytes")
        raw = ca.synth_deflate_payload(n * chunk - 17, chunk, seed=n)
        comp, blk, _, nc = ca.deflate_compress_chunks(raw, chunk, level=6)
        out, _ = ca.deflate.decompress_gpu(ctx, comp, blk, chunk)
        assert nc == n and out.tobytes() == raw.tobytes()
