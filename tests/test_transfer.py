"""The state transfers' chunks and threads (csrc/transfer.cpp) on the CPU."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "rkdg_heter_calculate_amd", "csrc")


def test_transfers_carry_every_byte_and_hold_what_they_need(tmp_path):
    exe = str(tmp_path / "transfer_check")
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-Wno-unused-function", "-I", os.path.join(ROOT, "tests", "stub_hip"), "-I", CSRC, "-o", exe,
                    os.path.join(ROOT, "tests", "transfer_check.cpp"), os.path.join(CSRC, "transfer.cpp"), "-lpthread"],
                   check=True)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stdout[-2000:]
