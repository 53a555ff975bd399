"""The strain limit's FP64 screen against its exact test (cs_strain_edge.h): no
decision may differ, whatever the lengths, and every edge farther than a few
1e-9 from the limits must be decided by it."""
import os
import subprocess

SRC = os.path.join(os.path.dirname(os.path.abspath(__file__)), "cpp", "strain_edge_test.cpp")


def test_screen_agrees_with_the_exact_test(tmp_path):
    exe = tmp_path / "edge"
    subprocess.run(["g++", "-std=c++17", "-O2", "-ffp-contract=off", "-o", str(exe), SRC], check=True)
    out = subprocess.run([str(exe)], check=True, capture_output=True, text=True).stdout
    cases, wrong, undecided = map(int, out.split())
    assert cases > 1_000_000 and wrong == 0 and undecided == 0
