"""The mask kernel's FP32 node tests are sound: built for the host and held
against their FP64 forms at the threshold."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_fp32_node_tests_are_sound(tmp_path):
    exe = tmp_path / "rel"
    subprocess.run(["g++", "-O2", "-std=c++17", "-ffp-contract=off", os.path.join(ROOT, "tests", "cpu_rel_bounds_check.cpp"),
                    "-o", str(exe)], check=True)
    cases, bad_s, bad_b, s64, s32, b64, b32 = map(int, subprocess.run([str(exe)], check=True, capture_output=True,
                                                                     text=True).stdout.split())
    assert bad_s == 0 and bad_b == 0
    assert s32 > cases // 10 and b32 > cases // 10  # and they do find nodes apart
