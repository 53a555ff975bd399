"""Long chains, laid out for the banded sweeps and for all sweeps in one
work-group: which of them runs follows the number of bonds over the limit, and
both end as the sequential model does.  Few bonds: the levels without one are
skipped."""
import numpy as np
import pytest

from collision_amd import scenes as S
from collision_amd.solver import solver_for_scene
from tests.test_gpu_strain_chains import sweeps

pytestmark = pytest.mark.gpu


def string(n, closed, moved):
    r = 0.1 * n / (2 * np.pi)
    t = 2 * np.pi * np.arange(n) / n
    x = np.stack([r * np.cos(t), r * np.sin(t), 0 * t], 1)
    v = np.zeros_like(x)
    g = np.random.default_rng(n)
    i = g.choice(n, moved, replace=False)
    along = np.stack([-np.sin(t), np.cos(t), 0 * t], 1)
    v[i] = along[i] * g.uniform(15.0, 25.0, (moved, 1)) * g.choice([-1.0, 1.0], (moved, 1))
    b = S._Builder()
    b.add_string(x, v)
    if closed:
        b.bonds[0] = np.concatenate([b.bonds[0], np.array([[n - 1, 0]], np.int32)])
    big = 2 * r + 10
    return b.build(f"string_{n}", thickness=1e-5, dt=1e-3, steps=1, domain_lo=(-big,) * 3,
                   domain_hi=(big,) * 3)


@pytest.mark.parametrize("sweeps_max", [10, 23])
@pytest.mark.parametrize("n,closed,moved", [(500, False, 2), (1000, False, 3), (4000, False, 3),
                                            (4000, False, 1500), (4000, True, 3), (4000, True, 1500),
                                            (70000, False, 3)])
def test_chain_matches_the_sequential_sweeps(n, closed, moved, sweeps_max):
    sc = string(n, closed, moved)
    av, done, last = sweeps(sc, sweeps_max)
    solver = solver_for_scene(sc, pass_timing=0, max_strain_sweeps=sweeps_max)
    for _ in range(2):  # (the second time from the state set again)
        solver.setState(sc.x, sc.vel)
        rep = solver.step()
        out = solver.getState()
        assert (rep.status, rep.hit_pairs) == (0, 0)
        assert (rep.strain_sweeps, rep.strain_edges) == (done, last) and done > 1
        assert np.array_equal(out["avg_vel"], av)
        if moved < 10 and 512 < n - (not closed) <= 65536:
            assert rep.strain_levels < done * n // 2  # (the bands go through all of every sweep)
    solver.close()
