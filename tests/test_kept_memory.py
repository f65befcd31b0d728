"""Memory the library keeps between calls (default-stream scratch, host-to-host calls): sizes
that grow and shrink, threads that share the default stream, gst_free_decompressor between
calls, and a call after one that failed."""
import threading

import numpy as np
import pytest

import gst_amd
from gst_amd import encode

from test_ans_chain import _encode

pytestmark = pytest.mark.gpu

SIZES = [(801, 512, 512), (802, 1024, 1024), (803, 512, 256), (804, 1920, 1024), (805, 768, 512)]


def _threads(n, body):
    errors = []

    def run(i):
        try:
            body(i)
        except BaseException as e:  # pytest's own failures too: reported by the test's thread
            errors.append(e)
    threads = [threading.Thread(target=run, args=(i,)) for i in range(n)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not errors


@pytest.mark.parametrize("stream", ["default", "created"])
def test_threads_share_a_stream(device, stream):
    torch = device.torch
    files, dxts = encode.make_textures(SIZES)
    staged = []
    for f in files:
        staging, (h,) = gst_amd.PackStaging([f])
        staged.append((h, device.upload(staging)))
    s = torch.cuda.default_stream() if stream == "default" else torch.cuda.Stream()
    device.sync()

    def body(i):
        order = np.random.default_rng(i).permutation(len(files))
        outs = [torch.full((h.dxt_bytes,), 0xA5, dtype=torch.uint8, device=device.dev) for h, _ in staged]
        torch.cuda.synchronize()
        for k in order:
            h, d_cmp = staged[k]
            gst_amd.LoadCompressedDXT(h, s.cuda_stream, d_cmp.data_ptr(), outs[k].data_ptr())
        s.synchronize()
        for o, d in zip(outs, dxts):
            assert o.cpu().numpy().tobytes() == d
        if i == 0:
            gst_amd.FreeDecompressor()
    _threads(6, body)
    assert gst_amd.ReadErrorBits(s.cuda_stream) == 0


def test_host_calls(device):
    files, dxts = encode.make_textures(SIZES)
    bad = bytearray(files[0])
    bad[28:30] = (int.from_bytes(bad[28:30], "little") + 3).to_bytes(2, "little")

    def body(i):
        for k in np.random.default_rng(i).permutation(len(files)):
            assert gst_amd.DecompressDXT(files[k]) == dxts[k]
            with pytest.raises(gst_amd.GstError) as e:
                gst_amd.DecompressDXT(bytes(bad))
            assert e.value.code == -3
            if i == 0:
                gst_amd.FreeDecompressor()
    _threads(6, body)


def test_ans_calls(device):
    norm = np.full(256, 8, np.int64)

    def body(i):
        rng = np.random.default_rng(i)
        d = gst_amd.AnsDecoder(norm.tolist(), 32)
        try:
            for groups in (1, 40, 3, 130):  # 130: more than the smallest kept buffer holds
                syms = rng.integers(0, 256, (groups, 32, 256))
                words, x = _encode(norm, syms)
                data = [w.astype("<u2").tobytes() for w in words]
                got = d.decode([int(v) for v in x.reshape(-1)], data)
                assert got == [s.astype(np.uint8).tobytes() for s in syms.reshape(-1, 256)]
                if i == 0:
                    gst_amd.FreeDecompressor()
        finally:
            d.close()
    _threads(3, body)
