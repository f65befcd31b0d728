"""The rANS kernels with two groups a wave, in every shape they are built in, on streams at
the edges of their rings: no renormalisation word at all, 16 words a step and 22 a step, for
group counts that leave a wave one group, none, or a short unit."""
import pytest

import gst_amd
from oracle import gst_oracle as go
from test_ans_chain import _texture

pytestmark = pytest.mark.gpu

SHAPES = [dict(ans_form="paired"), dict(ans_form="plain"), dict(waves_per_group=8)]
SHAPES += [dict(waves_per_group=w, groups_per_wave=g, separate_table_stage=True)
           for w, g in ((1, 2), (2, 1), (2, 2), (4, 1), (8, 2))]


@pytest.mark.parametrize("kind", ["constant", "uniform", "rare"])
def test_ring_edges_match_oracle(device, kind):
    files = [_texture(512, 256, 1, kind, 1), _texture(512, 512, 3, kind, 2), _texture(640, 1024, 6, kind, 4)]
    expected = []
    for f in files:
        rc, out, _ = go.decode_dxt(f, nthreads=8)
        assert rc == go.OK
        expected.append(out)
    hdrs = [gst_amd.ParseHeader(f) for f in files]
    d_files = [device.upload(f) for f in files]
    for shape in SHAPES:
        # A grid of 3: every work-group decodes many units in turn, with the rings reused.
        for grids in (None, {"ans_decode": 3}):
            outs = [device.empty(h.dxt_bytes) for h in hdrs]
            b = gst_amd.Batch(len(files), sum(h.num_blocks for h in hdrs), sum(h.palette_bytes for h in hdrs),
                              grids=grids, **shape)
            try:
                b.bind(hdrs, [t.data_ptr() for t in d_files], [t.data_ptr() for t in outs], device.stream)
                b.decode(device.stream)
                assert [device.download(o) for o in outs] == expected, shape
                assert b.error_bits(device.stream) == 0
            finally:
                b.close()
