"""bench.py's command line on a CPU-only host: more than one GPU is refused
with a message and a non-zero status, before anything touches a device."""
import os
import subprocess
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_more_than_one_gpu_is_refused():
    r = subprocess.run([sys.executable, os.path.join(ROOT, "bench.py"), "--gpus", "2"],
                       capture_output=True, text=True, timeout=120)
    assert r.returncode == 2
    assert "one GPU" in r.stderr and r.stdout == ""


@pytest.mark.parametrize("path,n,fused,faces,update", [
    ("tiled", (256, 264, 256), False, 4 * (8 + 11), 4 * (11 + 3 + 8 + 8)),
    ("tiled", (100, 85, 101), False, 4 * (8 + 11), 4 * (11 + 3 + 8 + 8)),
    ("tiled", (85, 100, 100), False, 4 * (8 + 21), 4 * (21 + 3 + 8 + 8)),
    ("tiled", (16, 24, 16), True, None, 4 * (8 + 8 + 8)),
    ("strict", (16, 24, 16), False, None, 4 * (21 + 3 + 8 + 8))])
def test_roofline_bytes_are_those_of_the_kernels_run(path, n, fused, faces, update):
    """Arrays read and written by the second stage's launches, by route."""
    sys.path.insert(0, ROOT)
    import bench
    launches = 0 if fused or path != "tiled" else 10
    b = bench.kernel_bytes(path, {"n": n}, {"faces_s1": (1.0, launches)})
    assert b.get("faces_s2") == faces and b["update_s2"] == update
