"""Host-to-host calls past the size that pinned memory is kept for: they go through ordinary
memory, and their results are the oracle's and those of smaller calls."""
import struct

import numpy as np
import pytest

from conftest import load_golden

import gst_amd
from oracle import gst_oracle as go

from test_ans_chain import _encode

pytestmark = pytest.mark.gpu


def _repeat(gtc, w, h):
    """A w x h texture whose planes repeat the rANS groups of `gtc`'s."""
    hdr = struct.unpack_from("<7I", gtc, 0)
    nv, times, at, parts = hdr[0] * hdr[1] // 16, w * h // (hdr[0] * hdr[1]), 28 + 2048, []
    for syms, size, planes in zip((2 * nv, 4 * nv, hdr[2], nv), hdr[3:], (2, 4, 1, 1)):
        ends = np.frombuffer(gtc, "<u4", syms // 8192, at)
        starts = np.concatenate([[4 * len(ends)], ends[:-1]])
        groups = [gtc[at + int(a):at + int(b)] for a, b in zip(starts, ends)]
        per = len(groups) // planes
        seq = [g for p in range(planes) for g in groups[p * per:(p + 1) * per] * times]
        parts.append((4 * len(seq) + np.cumsum([len(g) for g in seq])).astype("<u4").tobytes() + b"".join(seq))
        at += size
    return struct.pack("<7I", w, h, hdr[2] * times, *map(len, parts)) + gtc[28:28 + 2048] + b"".join(parts)


def test_decompress_dxt(device):
    piece = load_golden("ref_test1")["gtc"].tobytes()
    f = _repeat(piece, 16384, 8192)
    rc, expected, _ = go.decode_dxt(f, nthreads=8)
    assert rc == go.OK
    bad = bytearray(f)
    bad[28:30] = (int.from_bytes(bad[28:30], "little") + 3).to_bytes(2, "little")
    for _ in range(2):
        assert gst_amd.DecompressDXT(f) == expected
        with pytest.raises(gst_amd.GstError) as e:
            gst_amd.DecompressDXT(bytes(bad))
        assert e.value.code == -3
        assert gst_amd.DecompressDXT(piece) == load_golden("ref_test1")["dxt"].tobytes()


def test_ans_groups(device):
    norm = np.full(256, 8, np.int64)
    syms = np.random.default_rng(3).integers(0, 256, (4, 32, 256))
    words, x = _encode(norm, syms)
    data = [w.astype("<u2").tobytes() for w in words]
    states, expected = x.reshape(-1).tolist(), [s.astype(np.uint8).tobytes() for s in syms.reshape(-1, 256)]
    d = gst_amd.AnsDecoder(norm.tolist(), 32)
    try:
        assert d.decode(states, data) == expected
        assert d.decode(states * 2048, data * 2048) == expected * 2048
    finally:
        d.close()
