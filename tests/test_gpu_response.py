"""Hit sorting and the Jacobi apply against the oracle at chosen hit counts:
`count` pairs of crossing bonds give one hit and four records each, so the
hit and record sorts run at, below and above 64 keys and across the limit
between rank counting and radix passes (32,768 records)."""
import numpy as np
import pytest

from collision_amd import scenes as S
from tests.parity import run_parity

pytestmark = pytest.mark.gpu


def crossing_pairs(count):
    g = np.random.default_rng(count)
    side = int(np.ceil(np.sqrt(count)))
    at = np.stack([np.arange(count) % side, np.arange(count) // side], 1) * 0.05
    b = S._Builder()
    for upper in (0, 1):
        for i in g.permutation(count):  # the partners' ids are unrelated
            c = np.array([at[i, 0], at[i, 1], 4e-4 * upper])
            d = np.array([0.0, 0.01, 0.0]) if upper else np.array([0.01, 0.0, 0.0])
            v = np.array([0.0, 0.0, -0.3 if upper else 0.3])
            b.add_string(np.stack([c - d, c + d]), np.tile(v, (2, 1)) + 0.01 * g.normal(size=(2, 3)))
    big = 0.05 * side + 10.0
    return b.build(f"crossing_{count}", thickness=1e-3, dt=1e-3, steps=2, friction=0.2,
                   domain_lo=(-big,) * 3, domain_hi=(big,) * 3)


@pytest.mark.parametrize("count", [1, 15, 16, 17, 64, 65, 257, 8193])
def test_hits_match_the_oracle(count):
    st = run_parity(crossing_pairs(count), steps=2)
    assert st["hit_pairs"] >= count
