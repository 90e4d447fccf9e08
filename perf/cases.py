"""The calls by which this framework's decoders are timed.

Every case is one call of a public entry point of ``codag_amd`` on inputs that
already lie where its user has them: the compressed streams, their offsets and
the output buffer in device memory (a host buffer for the one synchronous
host-buffer case), encoded beforehand by the package's own producers or, for
single Deflate streams, by zlib.

Kinds of case:

* ``rlev1`` / ``rlev2``: an ORC integer column cut into chunks; ``source``
  ``synth`` is the benchmark column (RLE v1: runs and literal groups; RLE v2: a
  quarter each of SHORT_REPEAT, DIRECT, PATCHED_BASE and DELTA), ``column`` a
  table column (categories, counters, measurements) written by the encoder.
* ``chunks``: the Deflate chunk container.
* ``batch``: independent zlib or gzip streams of uneven size, largest first.
* ``brle`` / ``lzss``: the byte codecs' containers.
* ``rlev1_host``: ``rle_v1.decompress_gpu_orig``, host buffers in and out.
"""
import math
import random
import zlib
from concurrent.futures import ThreadPoolExecutor

import numpy as np
import torch

import codag_amd as ca

THREADS = 16
_ctx = None


def _context():
    """The one context that a program keeps."""
    global _ctx
    if _ctx is None:
        _ctx = ca.Context(torch.cuda.current_device())
    return _ctx


def listed():
    return [
        # a 128 MiB uint64 column of a table scan
        dict(name="rlev1_u64_128m", kind="rlev1", source="synth", width=8, values=1 << 24, chunk=131072),
        # a small column of one-byte codes, decoded from host buffers as the command line tool does
        dict(name="rlev1_host_u8_4m", kind="rlev1_host", source="column", width=1, values=(4 << 20) - 77, chunk=131072),
        # the wide and the common column type of an RLE v2 scan
        dict(name="rlev2_u64_256m", kind="rlev2", source="synth", width=8, values=1 << 25, chunk=131072),
        dict(name="rlev2_u32_184m", kind="rlev2", source="synth", width=4, values=48_123_457, chunk=131072),
        # one stripe of a narrow column: fewer chunks than the GPU has compute units
        dict(name="rlev2_u16_5m", kind="rlev2", source="column", width=2, values=2_600_011, chunk=131072),
        # a 512 MiB Deflate container, one of 32 MiB, and three chunks fetched by themselves
        dict(name="chunks_512m", kind="chunks", level=6, bytes=512 << 20, chunk=131072),
        dict(name="chunks_32m", kind="chunks", level=6, bytes=(32 << 20) - 12345, chunk=131072),
        dict(name="chunks_3", kind="chunks", level=9, bytes=3 * 131072 - 999, chunk=131072),
        # uneven streams of a file store (fixed, dynamic and stored blocks mixed), and small gzip members of a message log
        dict(name="batch_zlib_300", kind="batch", streams=300, lo=4 << 10, hi=4 << 20, format="zlib"),
        dict(name="batch_gzip_3000", kind="batch", streams=3000, lo=1 << 10, hi=64 << 10, format="gzip"),
        # byte columns: runs and literal stretches; text
        dict(name="brle_256m", kind="brle", bytes=256 << 20, chunk=262144),
        dict(name="lzss_256m", kind="lzss", bytes=(256 << 20) - 4321, chunk=131072),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["rlev1", "rlev2", "chunks", "chunks", "batch", "batch", "brle", "lzss", "rlev1_host"])
    if kind in ("rlev1", "rlev2", "rlev1_host"):
        width = rng.choice([1, 2, 4, 8])
        most = (16 << 20) if kind == "rlev1_host" else (128 << 20) if kind == "rlev1" else (256 << 20)
        return dict(kind=kind, source=rng.choice(["synth", "column"]), width=width,
                    values=_log(rng, 32768, most) // width, chunk=rng.choice([32768, 131072, 131072]))
    if kind == "chunks":
        return dict(kind=kind, level=rng.choice([1, 6, 6, 9]), bytes=_log(rng, 1 << 14, 512 << 20),
                    chunk=rng.choice([65536, 131072, 131072]))
    if kind == "batch":
        hi = _log(rng, 16 << 10, 4 << 20)
        return dict(kind=kind, streams=max(1, min(4000, _log(rng, 4 << 20, 192 << 20) // hi)),
                    lo=rng.choice([1 << 10, 4 << 10]), hi=hi, format=rng.choice(["zlib", "gzip"]))
    if kind == "brle":
        return dict(kind=kind, bytes=_log(rng, 1 << 16, 256 << 20), chunk=262144)
    return dict(kind=kind, bytes=_log(rng, 1 << 16, 256 << 20), chunk=131072)


def _column(n, width, seed):
    """n values of a table column: stretches of repeated categories, counters and
    measurements around a level, a few thousand values each."""
    g = np.random.default_rng(seed)
    top = 1 << (8 * width - 1)
    parts, have = [], 0
    while have < n:
        m = int(g.integers(1000, 60000))
        what = int(g.integers(0, 3))
        if what == 0:
            k = m // 8 + 1
            p = np.repeat(g.zipf(1.6, k) % min(top, 5000), g.geometric(0.12, k))[:m]
        elif what == 1:
            p = int(g.integers(0, top)) + np.cumsum(g.integers(0, int(g.integers(2, 40)), m))
        else:
            p = int(g.integers(0, top)) + g.integers(0, min(top, 1 << int(g.integers(3, 20))), m)
            p[:: int(g.integers(50, 300))] += int(g.integers(0, min(top, 1 << 30)))
        parts.append(p.astype(np.uint64))
        have += len(p)
    return np.concatenate(parts)[:n].astype("u%d" % width)


def _rle(case, seed):
    """(compressed bytes, offsets, lengths, chunk count, the container as written)"""
    v1 = case["kind"] != "rlev2"
    n, w, ch = case["values"], case["width"], case["chunk"]
    if case["source"] == "synth":
        if v1:
            _, cont, off, ln, nc = ca.synth_rlev1(n, w, ch, min(1 << 16, 1 << (8 * w)), seed=seed + 1)
        else:
            _, cont, off, ln, nc = ca.synth_rlev2(n, w, ch, seed=seed + 1)
    else:
        cont, off, ln, nc = (ca.rlev1_encode if v1 else ca.rlev2_encode)(_column(n, w, seed), w, ch)
    return cont[8:] if v1 else cont, off[:nc], ln[:nc], nc, (cont, off, ln)


def _stream_sizes(case):
    r = random.Random(case["streams"] * 31 + case["hi"])
    lo, hi = min(case["lo"], case["hi"]), case["hi"]
    return sorted((_log(r, lo, hi) for _ in range(case["streams"])), reverse=True)


def _payloads(case, seed):
    sizes = _stream_sizes(case)
    raw = ca.synth_deflate_payload(sum(sizes), 32768, seed=seed + 1)
    at = np.concatenate([[0], np.cumsum(sizes)])
    return [raw[at[i]:at[i + 1]] for i in range(len(sizes))]


def _streams(case, seed):
    def one(i):
        p = parts[i]
        if case["format"] == "gzip":
            c = zlib.compressobj(6, zlib.DEFLATED, 31)
            return np.frombuffer(c.compress(p) + c.flush(), np.uint8)
        return ca.deflate_compress_mixed(p, 20, 5, 32768, seed=seed + i)[0]

    parts = _payloads(case, seed)
    with ThreadPoolExecutor(THREADS) as ex:
        return list(ex.map(one, range(len(parts))))


def _chunk_container(case, seed):
    raw = ca.synth_deflate_payload(case["bytes"], case["chunk"], seed=seed + 1)
    return ca.deflate_compress_chunks(raw, case["chunk"], level=case["level"], threads=THREADS)


def _dev(a):
    return torch.from_numpy(np.array(a, copy=True)).cuda()


def _addr(t):
    return t.data_ptr()


def prepare(case, seed):
    kind = case["kind"]
    s = dict(case=case, ctx=_context())
    if kind == "rlev1_host":
        _, _, _, n, s["files"] = _rle(case, seed)
        return s
    if kind in ("rlev1", "rlev2"):
        comp, off, ln, n, _ = _rle(case, seed)
        s.update(off=_dev(off.view(np.int64)), len=_dev(ln.view(np.int64)))
        out = n * case["chunk"]
    elif kind == "chunks":
        comp, blk, _, n = _chunk_container(case, seed)
        s.update(off=_dev(blk[1:].view(np.int64)))
        out = n * case["chunk"]
    elif kind == "batch":
        streams, sizes = _streams(case, seed), _stream_sizes(case)
        n = len(streams)
        # every stream and every output begins on a 16-byte boundary, as an allocator would place them
        s_at = np.concatenate([[0], np.cumsum([(len(x) + 15) // 16 * 16 for x in streams])])
        o_at = np.concatenate([[0], np.cumsum([(x + 15) // 16 * 16 for x in sizes])])
        comp = np.zeros(int(s_at[-1]), np.uint8)
        for a, x in zip(s_at, streams):
            comp[a:a + len(x)] = x
        out = int(o_at[-1])
    elif kind == "brle":
        raw = ca.synth_byte_payload(case["bytes"], 0, seed=seed + 1)
        comp, idx, _ = ca.brle_container(ca.brle_encode(raw, case["chunk"], THREADS))
        n = len(idx) - 1
        s.update(off=_dev(np.array(idx).view(np.int64)))
        out = n * case["chunk"]
    else:
        raw = ca.synth_byte_payload(case["bytes"], 1, seed=seed + 1)
        comp, idx, _, _ = ca.lzss_container(ca.lzss_encode(raw, case["chunk"], THREADS))
        n = len(idx)
        s.update(off=_dev(np.array(idx).view(np.int64)))
        out = n * case["chunk"]
    s.update(n=n, comp=_dev(comp), comp_bytes=len(comp), out=torch.zeros(out, dtype=torch.uint8, device="cuda"),
             status=torch.zeros(n, dtype=torch.int32, device="cuda"),
             out_len=torch.zeros(n, dtype=torch.int64, device="cuda"))
    if kind == "batch":
        d = np.zeros((n, 4), np.int64)
        d[:, 0] = _addr(s["comp"]) + s_at[:-1]
        d[:, 1] = [len(x) for x in streams]
        d[:, 2] = _addr(s["out"]) + o_at[:-1]
        d[:, 3] = sizes
        s.update(descs=_dev(d), results=torch.zeros((n, 2), dtype=torch.int64, device="cuda"))
    torch.cuda.synchronize()  # the decoders run on the context's own stream
    return s


def run(s):
    case, ctx = s["case"], s["ctx"]
    kind = case["kind"]
    if kind == "rlev1_host":
        cont, off, ln = s["files"]
        return ca.rle_v1.decompress_gpu_orig(ctx, cont, off, ln, case["width"], case["chunk"])[0]
    if kind == "batch":
        flags = ca.INFLATE_GZIP if case["format"] == "gzip" else 0
        ctx.inflate_batch(_addr(s["descs"]), s["n"], _addr(s["results"]), flags)
        return {"out": s["out"], "results": s["results"]}
    comp, out, st, n, ch = _addr(s["comp"]), _addr(s["out"]), _addr(s["status"]), s["n"], case["chunk"]
    if kind in ("rlev1", "rlev2"):
        decode = ctx.rlev1_decode if kind == "rlev1" else ctx.rlev2_decode
        decode(comp, s["comp_bytes"], _addr(s["off"]), _addr(s["len"]), n, case["width"], ch, out, st)
        return {"out": s["out"], "status": s["status"]}
    if kind == "chunks":
        ctx.inflate_chunks(comp, s["comp_bytes"], _addr(s["off"]), n, ch, out, _addr(s["out_len"]), st)
    else:
        decode = ctx.brle_decode if kind == "brle" else ctx.lzss_decode
        decode(comp, s["comp_bytes"], _addr(s["off"]), n, ch, out, _addr(s["out_len"]), st)
    return {"out": s["out"], "status": s["status"], "out_len": s["out_len"]}


def _out_bytes(case):
    if case["kind"] == "batch":
        return sum(_stream_sizes(case))
    if "values" in case:
        return case["values"] * case["width"]
    return case["bytes"]


# compressed bytes per output byte, about what the producers reach on these inputs
_RATIO = {"chunks": 0.48, "batch": 0.54, "brle": 0.55, "lzss": 0.66}
_RLE_RATIO = {8: 0.25, 4: 0.27, 2: 0.5, 1: 1.0}


def work(case):
    out = _out_bytes(case)
    ratio = _RATIO[case["kind"]] if case["kind"] in _RATIO else _RLE_RATIO[case["width"]]
    return {"bytes": out * (1 + ratio), "flops": 0}


def exact(case, seed):
    """The decoded streams by zlib itself; None for the codecs that only this package has."""
    kind = case["kind"]
    if kind == "chunks":
        comp, blk, _, n = _chunk_container(case, seed)
        off, ch = blk[1:].astype(np.int64), case["chunk"]
        out = np.zeros(n * ch, np.uint8)

        def one(i):
            raw = zlib.decompressobj().decompress(memoryview(comp[off[i]:off[i + 1]]))
            out[i * ch:i * ch + len(raw)] = np.frombuffer(raw, np.uint8)
            return len(raw)

        with ThreadPoolExecutor(THREADS) as ex:
            lens = list(ex.map(one, range(n)))
        return {"out": out, "status": np.zeros(n, np.int32), "out_len": np.array(lens, np.int64)}
    if kind == "batch":
        streams, sizes = _streams(case, seed), _stream_sizes(case)
        at = np.concatenate([[0], np.cumsum([(x + 15) // 16 * 16 for x in sizes])])
        out, res = np.zeros(int(at[-1]), np.uint8), np.zeros((len(streams), 2), np.int64)
        check = zlib.crc32 if case["format"] == "gzip" else zlib.adler32
        for i, x in enumerate(streams):
            raw = zlib.decompress(memoryview(x), 47)
            out[at[i]:at[i] + len(raw)] = np.frombuffer(raw, np.uint8)
            res[i] = len(raw), np.array([check(raw) << 32], np.uint64).view(np.int64)[0]
        return {"out": out, "results": res}
    return None
