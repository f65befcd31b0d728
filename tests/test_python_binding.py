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
