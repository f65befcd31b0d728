"""Error bits read inside a graph that the caller captured: every replay gives its own."""
import ctypes

import pytest

from conftest import load_golden

import gst_amd

pytestmark = pytest.mark.gpu


def test_every_replay_reads_its_own_bits(device):
    torch = device.torch
    good = load_golden("ref_c0")["gtc"].tobytes()
    bad = bytearray(good)
    bad[28:30] = (int.from_bytes(bad[28:30], "little") + 3).to_bytes(2, "little")
    h = gst_amd.ParseHeader(good)
    d_good, d_bad = device.upload(good), device.upload(bytes(bad))
    d_file, d_out = d_good.clone(), device.empty(h.dxt_bytes)
    host = torch.zeros(1, dtype=torch.int32, pin_memory=True)
    fn = gst_amd.lib().gst_batch_error_bits_async
    fn.argtypes = [ctypes.c_void_p, ctypes.c_void_p, ctypes.c_void_p]
    b = gst_amd.Batch(1, h.num_blocks, h.palette_bytes)
    try:
        b.bind([h], [d_file.data_ptr()], [d_out.data_ptr()], device.stream)
        b.decode(device.stream)
        assert b.error_bits(device.stream) == 0
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=device.side):
            b.decode(device.stream)
            assert fn(b._h, device.stream, host.data_ptr()) == 0
        for i, data in enumerate((d_good, d_bad, d_good, d_bad, d_bad, d_good, d_good)):
            d_file.copy_(data)
            device.poison(d_out)
            host.fill_(-1)
            graph.replay()
            device.sync()
            assert (host.item() & 0x2 != 0) == (data is d_bad), "replay %d" % i
            assert data is d_bad or device.download(d_out) == load_golden("ref_c0")["dxt"].tobytes()
        assert b.error_bits(device.stream) == 0
    finally:
        b.close()
