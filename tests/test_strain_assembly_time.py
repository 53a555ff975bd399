"""Assembling a mesh whose elements have no locality (no banded strain plan fits)
computes the elements' levels once: the rest, a plan that does not fit and the
other schedule, takes less than they do."""
import os
import subprocess

from collision_amd import build as B

SRC = os.path.join(os.path.dirname(os.path.abspath(__file__)), "cpp", "strain_assembly_time.cpp")


def test_levels_are_computed_once(tmp_path):
    exe = tmp_path / "assembly"
    csrc = os.path.join(B.HERE, "csrc")
    subprocess.run([B.HIPCC, *B.COMMON_FLAGS, "-w", "-I", csrc, "-x", "hip", SRC,
                    os.path.join(csrc, "cs_schedule.hip"), "-o", str(exe)], check=True,
                   capture_output=True)
    out = subprocess.run([str(exe), "300"], check=True, capture_output=True, text=True).stdout
    levels, rest = map(float, out.split())
    assert rest < 0.6 * levels
