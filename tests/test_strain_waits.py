"""The banded strain sweep's waits against the bound after which the kernel gives
them up.  Where a vertex's visits span all levels (a closed string, a fan) each
sweep begins when the one before it is nearly over, so the tasks of the tenth
wait for nine sweeps, however long these are."""
import os
import subprocess

import pytest

SRC = os.path.join(os.path.dirname(os.path.abspath(__file__)), "cpp", "strain_wait_bound.cpp")


@pytest.fixture(scope="module")
def exe(tmp_path_factory):
    out = tmp_path_factory.mktemp("strain_waits") / "bound"
    subprocess.run(["g++", "-std=c++17", "-O2", "-o", str(out), SRC], check=True)
    return out


@pytest.mark.parametrize("mesh,n", [("ring", 3), ("ring", 1000), ("ring", 1 << 20), ("fan", 300000),
                                    ("grid", 64), ("grid", 512)])
def test_bound_covers_the_longest_wait(exe, mesh, n):
    out = subprocess.run([str(exe), mesh, str(n)], check=True, capture_output=True, text=True)
    steps, longest, bound = map(int, out.stdout.split())
    if mesh != "grid":
        assert longest >= 9 * (n - 3)  # (the serial case is the one tested)
    assert bound > longest
    # a broken plan is still reported: after seconds on an ordinary mesh
    assert bound < 2_000_000 or steps > 100_000
