"""The rANS kernel with a wave per group (the default for images and batches of few groups)
on streams at the edges of its ring: no renormalisation word at all, 16 words a step, and 22
a step (one more than a chunk every 12 steps), for group counts of every remainder; and the
stand-alone groups, which decode the same way."""
import struct

import numpy as np
import pytest

import gst_amd
from oracle import gst_oracle as go

pytestmark = pytest.mark.gpu


def _encode(norm, syms):
    """rANS over groups x streams x 256 symbols: (words of each group, final states)."""
    f, cum = norm[syms], (np.cumsum(norm) - norm)[syms]
    x = np.full(syms.shape[:2], 1 << 15, np.int64)
    words = [[] for _ in syms]
    for i in range(256):
        over = x >= f[:, :, i] << 20
        for g in np.flatnonzero(over.any(1)):
            words[g].append(x[g][over[g]] & 0xFFFF)
        x = np.where(over, x >> 16, x)
        x = (x // f[:, :, i] << 11) + x % f[:, :, i] + cum[:, :, i]
    return [np.concatenate(w) if w else np.zeros(0, np.int64) for w in words], x


def _stream(norm, syms):
    """One .gtc stream: u32 end offsets, then per group its words (padded in front to 4
    bytes) and 32 final states."""
    words, x = _encode(norm, syms)
    parts = []
    for g, w in enumerate(words):
        parts.append(np.concatenate([np.zeros(len(w) % 2, np.int64), w]).astype("<u2").tobytes() +
                     x[g].astype("<u4").tobytes())
    ends = 4 * len(parts) + np.cumsum([len(p) for p in parts])
    return ends.astype("<u4").tobytes() + b"".join(parts)


def _symbols(kind, rng, shape):
    if kind == "constant":
        norm = np.zeros(256, np.int64)
        norm[77] = 2048
        return norm, np.full(shape, 77)
    if kind == "uniform":
        return np.full(256, 8, np.int64), rng.integers(0, 256, shape)
    return np.array([1793] + [1] * 255, np.int64), rng.integers(1, 256, shape)  # rare: 11 bits a symbol


def _texture(width, height, palette_groups, kind, seed):
    rng = np.random.default_rng(seed)
    groups = width * height // 131072

    streams = [_symbols(kind, rng, (n, 32, 256)) for n in (2 * groups, 4 * groups, palette_groups)]
    if kind == "constant":
        norm = np.zeros(256, np.int64)
        norm[128] = 2048
        streams.append((norm, np.full((groups, 32, 256), 128)))
    else:
        idx = rng.integers(0, 100, groups * 8192)
        diff = np.diff(idx, prepend=0) + 128
        norm = np.array(gst_amd.NormalizeFrequencies(np.bincount(diff, minlength=256)), np.int64)
        streams.append((norm, diff.reshape(groups, 32, 256)))
    parts = [_stream(norm, syms) for norm, syms in streams]
    freqs = b"".join(norm.astype("<u2").tobytes() for norm, _ in streams)
    return struct.pack("<7I", width, height, 8192 * palette_groups, *map(len, parts)) + freqs + b"".join(parts)


@pytest.mark.parametrize("kind", ["constant", "uniform", "rare"])
def test_ring_edges_match_oracle(device, kind):
    files = [_texture(512, 256, 1, kind, 1), _texture(512, 512, 3, kind, 2), _texture(768, 512, 4, kind, 3),
             _texture(640, 1024, 6, kind, 4)]
    expected = []
    for f in files:
        rc, out, _ = go.decode_dxt(f, nthreads=8)
        assert rc == go.OK
        expected.append(out)
    for f, e in zip(files, expected):
        assert gst_amd.DecompressDXT(f) == e
    hdrs = [gst_amd.ParseHeader(f) for f in files]
    d_files = [device.upload(f) for f in files]
    # A grid of 3: every work-group decodes many units in turn, with the ring reused.
    for grids in (None, {"ans_decode": 3}):
        outs = [device.empty(h.dxt_bytes) for h in hdrs]
        b = gst_amd.Batch(len(files), sum(h.num_blocks for h in hdrs), sum(h.palette_bytes for h in hdrs),
                          grids=grids)
        try:
            b.bind(hdrs, [t.data_ptr() for t in d_files], [t.data_ptr() for t in outs], device.stream)
            b.decode(device.stream)
            assert [device.download(o) for o in outs] == expected
            assert b.error_bits(device.stream) == 0
        finally:
            b.close()


@pytest.mark.parametrize("kind", ["uniform", "rare"])
@pytest.mark.parametrize("groups,streams", [(1, 1), (3, 2), (4, 31), (5, 32), (9, 24)])
def test_stand_alone_groups(device, kind, groups, streams):
    norm, syms = _symbols(kind, np.random.default_rng(groups), (groups, streams, 256))
    words, x = _encode(norm, syms)
    data = [w.astype("<u2").tobytes() for w in words]
    d = gst_amd.AnsDecoder(norm.tolist(), streams)
    try:
        expected = [s.astype(np.uint8).tobytes() for s in syms.reshape(-1, 256)]
        assert d.decode(x.reshape(-1).tolist(), data) == expected
    finally:
        d.close()
