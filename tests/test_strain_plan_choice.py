"""The banded strain sweeps are for element orders with locality; where every band
meets most vertices the bands would run one after another, and all sweeps run in
one work-group."""
import os
import subprocess

import pytest

SRC = os.path.join(os.path.dirname(os.path.abspath(__file__)), "cpp", "strain_plan_choice.cpp")


@pytest.fixture(scope="module")
def exe(tmp_path_factory):
    out = tmp_path_factory.mktemp("strain_plan_choice") / "choice"
    subprocess.run(["g++", "-std=c++17", "-O2", "-o", str(out), SRC], check=True)
    return out


@pytest.mark.parametrize("n,kind,pays", [
    (2, "rows", 1), (16, "rows", 1), (64, "rows", 1), (256, "rows", 1), (64, "cols", 1), (256, "cols", 1),
    (64, "radial", 1), (256, "radial", 1), (64, "tiles16", 1), (160, "tiles16", 1), (128, "tiles64", 1),
    (64, "within256", 1), (96, "within1024", 1), (16, "random", 1), (24, "random", 1), (40, "random", 0), (64, "random", 0),
    (160, "random", 0), (200, "random", 0), (128, "tiles4", 0), (96, "within4096", 0)])
def test_choice_follows_the_order(exe, n, kind, pays):
    out = subprocess.run([str(exe), str(n), kind], check=True, capture_output=True, text=True)
    fits, got, imports, window = out.stdout.split()
    assert int(got) == pays, (imports, window)
    if (n, kind) == (96, "within1024"):  # (the banded path with a large window)
        assert int(window) > 65536
