"""The FP64 form's triangle-pair classification is sound: built for the host
and held against the reference's distance on pairs at the hit threshold."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_fp64_classification_is_sound(tmp_path):
    exe = tmp_path / "cull64"
    subprocess.run(["g++", "-O2", "-std=c++17", "-ffp-contract=off", os.path.join(ROOT, "tests", "cpu_cull64_check.cpp"),
                    "-o", str(exe)], check=True)
    cases, viol, miss, two, hits = map(int, subprocess.run([str(exe)], check=True, capture_output=True,
                                                           text=True).stdout.split())
    assert viol == 0
    assert miss > cases // 10 and two > cases // 100 and hits > cases // 5
