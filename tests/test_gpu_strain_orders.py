"""Strain sweeps against the oracle for element orders on both sides of the choice
between the banded sweeps and all sweeps in one work-group: rows shuffled within
1,024 elements (banded, a vertex window above 64 KB of LDS), columns, and random
orders just past the choice and far from it."""
import numpy as np
import pytest

from collision_amd import scenes as S
from tests.parity import run_parity

pytestmark = pytest.mark.gpu


def reordered(n, kind):
    sc = S.self_collision_cloth(n=n, name=f"{kind}_{n}")
    g = np.random.default_rng(3)
    if kind == "within1024":
        p = np.argsort(np.arange(sc.nt) + g.uniform(0, 1024, sc.nt), kind="stable")
    elif kind == "columns":
        c = sc.x[sc.tris].mean(1)
        p = np.lexsort((c[:, 1], np.round(c[:, 0], 6)))
    else:
        p = g.permutation(sc.nt)
    sc.tris, sc.tri_len0 = sc.tris[p], sc.tri_len0[p]
    return sc


@pytest.mark.parametrize("n,kind,steps", [(96, "within1024", 2), (64, "columns", 3), (16, "random", 4),
                                          (32, "random", 4), (96, "random", 2)])
def test_sweeps_match_the_oracle(n, kind, steps):
    st = run_parity(reordered(n, kind), steps=steps)
    assert st["strain_sweeps"] > steps
