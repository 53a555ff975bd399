"""The launch-shape tuner's scores: a candidate is judged by the launches it
reaches and by no others."""
import os
import subprocess

SRC = os.path.join(os.path.dirname(os.path.abspath(__file__)), "cpp", "launch_tuner_test.cpp")


def test_choices_follow_the_launches_they_reach(tmp_path):
    exe = tmp_path / "tuner"
    subprocess.run(["g++", "-std=c++17", "-O2", "-o", str(exe), SRC], check=True)
    p = subprocess.run([str(exe)], capture_output=True, text=True)
    assert p.returncode == 0, p.returncode
