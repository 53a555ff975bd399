"""The strain plan's records of long single strings take no more memory than the
records of the one-work-group sweep (a step of one element once took 2 KB)."""
import os
import subprocess

import pytest

SRC = os.path.join(os.path.dirname(os.path.abspath(__file__)), "cpp", "strain_plan_size.cpp")


@pytest.fixture(scope="module")
def exe(tmp_path_factory):
    out = tmp_path_factory.mktemp("strain_plan_size") / "size"
    subprocess.run(["g++", "-std=c++17", "-O2", "-o", str(out), SRC], check=True)
    return out


@pytest.mark.parametrize("n", [64, 1000, 1 << 20])
def test_records_of_a_string_stay_small(exe, n):
    out = subprocess.run([str(exe), str(n)], check=True, capture_output=True, text=True)
    records, before = map(int, out.stdout.split())
    assert records <= before
