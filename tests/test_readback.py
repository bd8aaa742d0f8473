"""Device memory to host memory through the pinned ring (cavs_amd/host/readback.cc): over a stand-in for the device
(tests/native/readback_check.cc) reads beyond the ring, two readers at a time, copies and waits that fail, no threads or
no pinned memory to be had; once more under the thread sanitizer.  Host only: no GPU."""
import os
import subprocess

import pytest

from cavs_amd import build

HERE = os.path.dirname(os.path.abspath(__file__))


def _check(tmp_path, flags, args):
    exe = str(tmp_path / "readback_check")
    src = [os.path.join(HERE, "native", "readback_check.cc"), os.path.join(build.HOST, "readback.cc")]
    subprocess.run([build.CXX] + build.CXX_FLAGS + flags + src + ["-ldl", "-o", exe], check=True, capture_output=True)
    return subprocess.run([exe] + args, capture_output=True, text=True, timeout=100)


@pytest.mark.parametrize("mode", [[], ["threadless"], ["ringless"]], ids=lambda m: m[0] if m else "plain")
def test_reads_through_the_ring(tmp_path, mode):
    r = _check(tmp_path, [], mode)
    assert r.returncode == 0, r.stdout + r.stderr


def test_reads_through_the_ring_under_the_thread_sanitizer(tmp_path):
    r = _check(tmp_path, ["-fsanitize=thread", "-g", "-DCHECK_UNDER_TSAN"], ["quick"])
    assert r.returncode == 0 and "WARNING" not in r.stderr, r.stdout + r.stderr
