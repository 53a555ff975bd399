"""Broad phase against the oracle on both sides of the element count from which
the full traversal has split rounds (4,096: below it no share of a walk has more
nodes than a walk may take)."""
import pytest

from tests.parity import run_parity
from tests.test_gpu_broad import loose_bonds

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("full", [0, 1], ids=["incremental", "full"])
@pytest.mark.parametrize("count,spread", [(4095, 0.35), (4096, 0.35)])
def test_candidates_match_the_oracle(count, spread, full):
    run_parity(loose_bonds(count, spread), steps=2, gpu_kw=dict(force_full_passes=full))
