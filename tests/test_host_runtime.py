"""The library's host code on a stand-in for the HIP runtime (CPU only; built by
gst_amd/build.py): what a call leaves behind it on the null stream, and what it does when the
runtime refuses it something or a wait fails."""
import os
import subprocess

import pytest

from conftest import ROOT

EXE = os.path.join(ROOT, "tests", "cpp", "host_runtime_test")


@pytest.mark.parametrize("check", ["batch_plan", "batch_error_bits", "stream_error_bits", "server_flags",
                                   "pinned_after_failed_wait", "no_pinned_memory", "little_device_memory",
                                   "large_host_calls", "async_error_bits", "little_lds"])
def test_host_code(check):
    proc = subprocess.run([EXE, check], capture_output=True, text=True, timeout=60)
    assert proc.returncode == 0, proc.stdout + proc.stderr
