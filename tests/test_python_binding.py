"""What the Python package leaves in the process that imports and calls it (CPU only)."""
import subprocess
import sys

from conftest import ROOT


def _run(code):
    proc = subprocess.run([sys.executable, "-c", code], cwd=ROOT, capture_output=True, text=True, timeout=120)
    assert proc.returncode == 0, proc.stdout + proc.stderr


def test_import_leaves_ctypes_pythonapi_alone():
    _run("""
import ctypes
before = ctypes.pythonapi.PyBytes_FromStringAndSize
was = (before.restype, before.argtypes)
import gst_amd
after = ctypes.pythonapi.PyBytes_FromStringAndSize
assert (after.restype, after.argtypes) == was
assert len(gst_amd._new_bytes(5)) == 5 and gst_amd._new_bytes(0) == b""
""")


def test_ans_decode_keeps_nothing():
    _run("""
import ctypes, tracemalloc
import gst_amd

class Library:
    @staticmethod
    def gst_ans_decode(handle, states, n, data, lens, n_data, raw):
        ctypes.memmove(raw, bytes(i % 251 for i in range(len(raw))), len(raw))
        return 0

gst_amd.lib = lambda: Library
d = gst_amd.AnsDecoder.__new__(gst_amd.AnsDecoder)
d._h = None
for n in (1, 31, 32, 33, 63, 64, 65, 127, 128, 768):
    got = d.decode([0] * n, b"")
    assert len(got) == n and {type(g) for g in got} == {bytes}
    assert b"".join(got) == bytes(i % 251 for i in range(256 * n))
del got
tracemalloc.start()
for n in range(2000, 2040):
    d.decode([0] * n, b"")
kept = tracemalloc.get_traced_memory()[0]
assert kept < 200000, kept
""")
