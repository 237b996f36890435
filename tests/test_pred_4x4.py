"""The SATD screening predicts a 4x4 at a time (pred_4x4, av1gpu_amd/csrc/av1m_common.h).  tests/cpp/pred_4x4_check.cpp (host
build) shows it equal to pred_px, which the spec's arithmetic defines, for every mode, angle, block size and 4x4."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_pred_4x4_equals_pred_px(tmp_path):
    exe = str(tmp_path / "pred_4x4_check")
    subprocess.run(["g++", "-O2", "-std=c++17", "-o", exe, os.path.join(ROOT, "tests", "cpp", "pred_4x4_check.cpp")], check=True)
    r = subprocess.run([exe], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout + r.stderr
    assert r.stdout.split()[0] == "ok" and int(r.stdout.split()[1]) > 1_000_000
