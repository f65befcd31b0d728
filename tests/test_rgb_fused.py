"""RGB8 output from the kernel that also holds the wavelet and the index scan: one tile a
row, odd tiles a row (pairs of tile positions straddle rows), coefficients whose colours
leave the byte range, palette indices outside the palette, and an output that is only
4-byte aligned."""
import numpy as np
import pytest

from conftest import load_golden

import gst_amd
from gst_amd import encode
from oracle import gst_oracle as go

pytestmark = pytest.mark.gpu


def _noisy(gtc, at, seed):
    """`gtc` with 200 bytes of noise in a stream's first renormalisation words."""
    b = bytearray(gtc)
    b[at:at + 200] = np.random.default_rng(seed).integers(0, 256, 200, dtype=np.uint8).tobytes()
    return bytes(b)


def _files():
    files, _ = encode.make_textures([(701, 128, 1024), (702, 640, 1024), (703, 768, 512), (704, 1024, 1024)])
    c0 = load_golden("ref_c0")["gtc"].tobytes()
    h = gst_amd.ParseHeader(c0)
    y = 28 + 2048 + 4 * (2 * h.num_blocks // 8192)
    chroma = 28 + 2048 + h.y_cmp_sz + 4 * (4 * h.num_blocks // 8192)
    palette = 28 + 2048 + h.y_cmp_sz + h.chroma_cmp_sz + 4 * (h.palette_bytes // 8192)
    return files + [_noisy(c0, y, 10), _noisy(c0, chroma, 11), _noisy(c0, palette, 13)]


@pytest.mark.parametrize("offset", [0, 4])
def test_rgb_matches_oracle(device, offset):
    files = _files()
    expected = []
    for f in files:
        rc, out = go.decode_rgb(f, nthreads=8)[:2]
        assert rc >= 0
        expected.append(out)
    for f, e in zip(files, expected):
        staging, (h,) = gst_amd.PackStaging([f])
        d_cmp, d_out = device.upload(staging), device.empty(3 * h.width * h.height + 16)
        gst_amd.LoadRGB(h, device.stream, d_cmp.data_ptr(), d_out.data_ptr() + offset)
        got = device.download(d_out)
        assert got[offset:offset + len(e)] == e
        assert got[:offset] == b"\xa5" * offset and got[offset + len(e):] == b"\xa5" * (16 - offset)
    gst_amd.ReadErrorBits(device.stream)  # the noisy palette's indices


def test_rgb_batch_equals_separate_kernels(device):
    files = _files()
    hdrs = [gst_amd.ParseHeader(f) for f in files]
    d_files = [device.upload(f) for f in files]
    got = []
    for separate in (False, True):
        outs = [device.empty(3 * h.width * h.height) for h in hdrs]
        b = gst_amd.Batch(len(files), sum(h.num_blocks for h in hdrs), sum(h.palette_bytes for h in hdrs),
                          rgb=True, separate_wavelet=separate, grids={"assemble": 11})
        try:
            b.bind(hdrs, [t.data_ptr() for t in d_files], [t.data_ptr() for t in outs], device.stream)
            b.decode(device.stream)
            got.append([device.download(o) for o in outs] + [b.error_bits(device.stream)])
        finally:
            b.close()
    assert got[0] == got[1]
