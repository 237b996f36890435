"""The quantizer divides by its step through the step's reciprocal and two exact corrections (quot_step,
av1gpu_amd/csrc/av1m_common.h).  tests/cpp/quot_check.cpp (host build) shows that the result is the IEEE quotient to the
bit for every step, over random magnitudes and around the thresholds the quantizer compares with."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_quot_step_is_the_ieee_quotient(tmp_path):
    exe = str(tmp_path / "quot_check")
    subprocess.run(["g++", "-O2", "-std=c++17", "-ffp-contract=off", "-mfma", "-o", exe, os.path.join(ROOT, "tests", "cpp", "quot_check.cpp")],
                   check=True)
    r = subprocess.run([exe], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout + r.stderr
    assert r.stdout.split()[0] == "ok" and int(r.stdout.split()[1]) > 10_000_000
