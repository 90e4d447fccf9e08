"""Edges of the LZSS decoder's parts, group batches, windows and segments: all
literals (9-byte groups, the most groups a part holds), all matches (17-byte
groups, output of several windows a step), mixtures, chunks of every small size
and streams cut anywhere. Compared with the oracle."""
import numpy as np
import pytest

import codag_amd as ca
import oracle
from tests.gpu_helpers import say

pytestmark = pytest.mark.gpu


def payload(kind, n):
    g = np.random.default_rng(n + len(kind))
    if kind == "noise":
        return g.integers(0, 256, n, dtype=np.uint8)
    if kind == "runs":
        return np.repeat(g.integers(0, 256, n // 3000 + 1, dtype=np.uint8), 3000)[:n]
    if kind == "period":
        return np.tile(g.integers(0, 256, 2046, dtype=np.uint8), n // 2046 + 1)[:n]
    return ca.synth_byte_payload(max(n, 1), 1, seed=n)[:n]


def decode(ctx, data, ends, chunk, out_bytes):
    n = len(ends)
    d_in = ctx.upload(np.concatenate([data, np.zeros(16, np.uint8)]))
    d_e, d_out = ctx.upload(np.asarray(ends, np.uint64)), ctx.alloc(n * chunk)
    d_len, d_st = ctx.alloc(8 * n), ctx.alloc(4 * n)
    d_out.fill(0xA5)
    ctx.lzss_decode(d_in, len(data), d_e, n, chunk, d_out, d_len, d_st)
    ctx.sync()
    return d_st.download(dtype=np.int32), d_len.download(dtype=np.uint64), d_out.download()


@pytest.mark.parametrize("kind", ["noise", "runs", "period", "text"])
@pytest.mark.parametrize("chunk", [1, 17, 1535, 1536, 1537, 6144, 6145, 131072])
def test_whole_chunks(kind, chunk):
    say(f"lzss: {kind}, chunks of {chunk}")
    raw = payload(kind, chunk * 3 + chunk // 2)
    data, ends, ch, orig = ca.lzss_container(ca.lzss_encode(raw, chunk))
    with ca.Context(0) as ctx:
        st, ln, out = decode(ctx, np.array(data), ends, chunk, orig)
    assert ch == chunk and not st.any()
    assert out[:orig].tobytes() == raw.tobytes() and int(ln.sum()) == orig
    assert (out[orig:] == 0xA5).all()


@pytest.mark.parametrize("kind", ["noise", "runs", "text"])
def test_cut_streams(kind):
    """One stream cut at every length around a step's parts: status, length and
    the bytes before the cut are the oracle's."""
    say(f"lzss: {kind}, cut streams")
    chunk = 40000
    raw = payload(kind, chunk)
    data, ends, _, _ = ca.lzss_container(ca.lzss_encode(raw, chunk))
    data = np.array(data)[: int(ends[0])]
    cuts = [c for c in (*range(1, 40), 207, 208, 209, 225, 3119, 3120, 3121, 3137, len(data) - 1, len(data)) if c <= len(data)]
    src = np.concatenate([data[:c] for c in cuts])
    e = np.cumsum(cuts).astype(np.uint64)
    want_st, want_len, want = oracle.lzss_decode_chunks(src, e, chunk)
    with ca.Context(0) as ctx:
        st, ln, out = decode(ctx, src, e, chunk, 0)
    assert (st == want_st).all() and (ln == want_len).all()
    for i in range(len(cuts)):
        k = int(ln[i])
        assert out[i * chunk:i * chunk + k].tobytes() == want[i * chunk:i * chunk + k].tobytes(), cuts[i]
        assert (out[i * chunk + k:(i + 1) * chunk] == 0xA5).all(), cuts[i]
