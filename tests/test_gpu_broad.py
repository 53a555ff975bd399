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


def loose_bonds(count, spread, length=0.02):
    """`count` single bonds at random places of a cube of edge `spread`"""
    g = np.random.default_rng(count)
    b = S._Builder()
    for _ in range(count):
        p = spread * g.random(3)
        b.add_string(np.stack([p, p + length * g.normal(size=3)]), g.normal(scale=0.5, size=(2, 3)))
    return b.build(f"loose_{count}", thickness=1e-3, dt=1e-3, steps=2)


@pytest.mark.parametrize("full", [0, 1], ids=["incremental", "full"])
@pytest.mark.parametrize("count,spread", [(1, 0.1), (2, 0.02), (255, 0.3), (256, 0.3), (257, 0.3),
                                          (513, 0.05), (1025, 0.4), (4097, 0.7),
                                          (32768, 1.5), (32769, 1.5)])
def test_candidates_match_the_oracle(count, spread, full):
    run_parity(loose_bonds(count, spread), steps=2, gpu_kw=dict(force_full_passes=full))


# The pair stream holds 3 n + 4,096 pairs at first and the first narrow launch
# covers max(n, 4,096) of them: streams below that, between the two (the rest is
# tested by a second launch) and above both (grown and walked again).
@pytest.mark.parametrize("full", [0, 1], ids=["incremental", "full"])
@pytest.mark.parametrize("count,range_", [(120, "below"), (200, "between"), (400, "above")])
def test_crowded_pair_streams_match_the_oracle(count, range_, full):
    scene = loose_bonds(count, 2.0, 2.0)
    x = np.asarray(scene.x).reshape(-1, 2, 3)
    lo, hi = x.min(1), x.max(1)
    over = ((lo[:, None] <= hi[None]) & (hi[:, None] >= lo[None])).all(2)
    pairs = int(np.triu(over, 1).sum())
    first, cap = max(count, 4096), 3 * count + 4096
    assert {"below": pairs < first - 50, "between": first + 50 < pairs < cap - 50,
            "above": pairs > cap + 50}[range_]
    run_parity(scene, steps=2, gpu_kw=dict(force_full_passes=full))
