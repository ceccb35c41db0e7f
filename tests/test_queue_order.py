"""The order in which the traversal's waves and the shading's blocks meet the
segments of a ray queue, compiled for the host from the kernels' own header
(tests/csrc/queue_check.cpp): complete, and even for every grid."""
import os
import shutil
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_segments_are_met_evenly(tmp_path):
    exe = str(tmp_path / "queue_check")
    r = subprocess.run([shutil.which("g++") or "g++", "-O2", "-std=c++17", "-o", exe,
                        os.path.join(ROOT, "tests", "csrc", "queue_check.cpp")], capture_output=True, text=True,
                       timeout=300)
    assert r.returncode == 0, r.stderr
    r = subprocess.run([exe], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0 and r.stdout.split() == ["cover", "0", "bad", "even", "0", "bad"], r.stdout
