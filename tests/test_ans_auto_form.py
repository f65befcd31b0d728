"""Batches on both sides of the line between the rANS kernel with a wave per group and the one
with work-groups of 8 groups of one stream (the unpaired form, which only batches of this size
take): streams at the edges of the rings, garbled streams and a bad frequency table, by launches
and by graphs captured with a small batch bound."""
import pytest

from conftest import load_golden

import gst_amd
from gst_amd import encode
from oracle import gst_oracle as go

from test_ans_chain import _texture
from test_batch import _garbled

pytestmark = pytest.mark.gpu


def _units(hdrs, per):
    return sum((g + per - 1) // per for h in hdrs for g in (
        2 * h.num_blocks // 8192, 4 * h.num_blocks // 8192, h.palette_bytes // 8192, h.num_blocks // 8192))


def _oracle(f):
    rc, out, _ = go.decode_dxt(f, nthreads=8)
    assert rc >= 0
    return out


def _decode_bad(device, f):
    """The blocks of a file with a bad frequency table, by the per-stream form."""
    h = gst_amd.ParseHeader(f)
    d_file, d_out = device.upload(f), device.empty(h.dxt_bytes)
    b = gst_amd.Batch(1, h.num_blocks, h.palette_bytes, ans_form="plain")
    try:
        b.bind([h], [d_file.data_ptr()], [d_out.data_ptr()], device.stream)
        b.decode(device.stream)
        assert b.error_bits(device.stream) & 0x2
        return device.download(d_out)
    finally:
        b.close()


def test_both_sides_of_the_line(device):
    cus = device.torch.cuda.get_device_properties(0).multi_processor_count
    c0 = load_golden("ref_c0")["gtc"].tobytes()
    special = [_texture(512, 256, 1, "constant", 1), _texture(512, 512, 3, "uniform", 2),
               _texture(640, 1024, 6, "rare", 4), c0, _garbled(c0, "y", 10), _garbled(c0, "chroma", 11)]
    bad = bytearray(c0)
    bad[28:30] = (int.from_bytes(bad[28:30], "little") + 3).to_bytes(2, "little")
    bad = bytes(bad)
    (filler,), (filler_dxt,) = encode.make_textures([(330, 1024, 1024)])
    expected = {f: _oracle(f) for f in special}
    expected[filler] = filler_dxt
    expected[bad] = _decode_bad(device, bad)

    hdr = gst_amd.ParseHeader
    fillers = (4 * cus - _units([hdr(f) for f in special], 4)) // _units([hdr(filler)], 4)
    below, above = special + [filler] * fillers, special + [bad] + [filler] * (fillers + 1)
    assert _units([hdr(f) for f in below], 4) <= 4 * cus < _units([hdr(f) for f in above], 4)
    assert _units([hdr(f) for f in above], 8) <= 6 * cus  # not paired
    hdrs = [hdr(f) for f in above]
    b = gst_amd.Batch(len(above), sum(h.num_blocks for h in hdrs), sum(h.palette_bytes for h in hdrs))
    try:
        for files in ([c0], below, above, below):
            hdrs = [hdr(f) for f in files]
            d_files = {f: device.upload(f) for f in set(files)}
            outs = [device.empty(h.dxt_bytes) for h in hdrs]
            b.bind(hdrs, [d_files[f].data_ptr() for f in files], [o.data_ptr() for o in outs], device.stream)
            b.capture_graph(device.stream)  # with the first bind; kept for the others
            for launch in (b.decode, b.launch_graph, b.launch_graph):
                for o in outs:
                    device.poison(o)
                launch(device.stream)
                for i, (f, o) in enumerate(zip(files, outs)):
                    assert device.download(o) == expected[f], "image %d of %d" % (i, len(files))
                assert b.error_bits(device.stream) == (0x2 if bad in files else 0)
    finally:
        b.close()
