"""Banded strain-limit sweeps against the oracle, at the edges of their plan:
one element, steps of 64 + 64 + 2 elements on one level, many bands that all
share vertices, a vertex window above 64 KB of LDS, and a mesh whose windows
do not fit at any band count (the one-work-group sweep)."""
import numpy as np
import pytest

from collision_amd import scenes as S
from tests.parity import run_parity

pytestmark = pytest.mark.gpu


def shuffled_cloth(n):
    """wavy cloth with its triangles in random order"""
    sc = S.self_collision_cloth(n=n, name=f"shuffled_{n}")
    p = np.random.default_rng(3).permutation(sc.nt)
    sc.tris, sc.tri_len0 = sc.tris[p], sc.tri_len0[p]
    return sc


def bonds(count, stretch=0.2):
    """`count` single bonds side by side, ends moving apart by `stretch` of their length a step"""
    b = S._Builder()
    for i in range(count):
        p = S.polyline((0.01 * i, 0.0, 0.0), (0.01 * i, 0.1, 0.0), 1)
        v = np.zeros_like(p)
        v[1, 1] = 0.1 * stretch / 1e-3
        b.add_string(p, v)
    return b.build(f"bonds_{count}", thickness=1e-4, dt=1e-3, steps=3)


@pytest.mark.parametrize("scene,steps", [(lambda: bonds(1), 3), (lambda: bonds(130), 3),
                                         (lambda: shuffled_cloth(24), 4), (lambda: shuffled_cloth(160), 2),
                                         (lambda: shuffled_cloth(200), 2)],
                         ids=["bond", "bonds130", "shuffled24", "shuffled160", "shuffled200"])
def test_banded_sweeps_match_the_oracle(scene, steps):
    st = run_parity(scene(), steps=steps, verbose=True)
    assert st["strain_sweeps"] > steps  # some step went on after its first sweep
