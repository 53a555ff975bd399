"""Broad phase against the oracle at the edges of its tiles: element counts
around the refit tile (256 leaves), one and several spanning nodes, walks cut
into the most and the fewest sub-ranges, and crowded elements whose
walks are long.  The candidate counts of every pass are compared
exactly (and everything else run_parity compares)."""
import numpy as np
import pytest

from collision_amd import scenes as S
from tests.parity import run_parity

pytestmark = pytest.mark.gpu


def loose_bonds(count, spread):
    """`count` single bonds at random places of a cube of edge `spread`"""
    g = np.random.default_rng(count)
    b = S._Builder()
    for _ in range(count):
        p = spread * g.random(3)
        b.add_string(np.stack([p, p + 0.02 * g.normal(size=3)]), g.normal(scale=0.5, size=(2, 3)))
    return b.build(f"loose_{count}", thickness=1e-3, dt=1e-3, steps=2)


@pytest.mark.parametrize("full", [0, 1], ids=["incremental", "full"])
@pytest.mark.parametrize("count,spread", [(1, 0.1), (2, 0.02), (255, 0.3), (256, 0.3), (257, 0.3),
                                          (513, 0.05), (1025, 0.4), (4097, 0.7)])
def test_candidates_match_the_oracle(count, spread, full):
    run_parity(loose_bonds(count, spread), steps=2, gpu_kw=dict(force_full_passes=full))
