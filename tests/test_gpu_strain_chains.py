"""Strain sweeps of a closed string against a sequential model: its first vertex
is met again by its last bond, so every sweep follows the whole of the one
before it and the kernel's waits last as long as the sweeps do."""
import heapq

import numpy as np
import pytest

from collision_amd import scenes as S
from collision_amd.solver import solver_for_scene

pytestmark = pytest.mark.gpu


def closed_string(n):
    r = 0.1 * n / (2 * np.pi)
    t = 2 * np.pi * np.arange(n) / n
    x = np.stack([r * np.cos(t), r * np.sin(t), 0 * t], 1)
    v = np.zeros_like(x)
    for i in (0, 1, n // 3, n // 2, n - 1):  # along the string, by a tenth to a third of a bond
        v[i] = (10.0 + 20.0 * i / n) * np.array([-np.sin(t[i]), np.cos(t[i]), 0.3])
    b = S._Builder()
    b.add_string(x, v)
    b.bonds[0] = np.concatenate([b.bonds[0], np.array([[n - 1, 0]], np.int32)])
    big = 2 * r + 10
    return b.build(f"closed_{n}", thickness=1e-4, dt=1e-3, steps=1, domain_lo=(-big,) * 3,
                   domain_hi=(big,) * 3)


def sweeps(sc, max_sweeps=10):
    """reduceSuperelast (dcollid.cpp:486-596) on the average velocities of one step, bonds in
    order; a bond is visited where an end changed since its last visit"""
    x, dt, n = sc.x, sc.dt, len(sc.bonds)
    av = ((x + dt * sc.vel) - x) / dt
    i, j = sc.bonds.T

    def over(a, b, va, vb, len0):
        def length(p, q):
            d = p - q
            return np.sqrt((d[..., 0] * d[..., 0] + d[..., 1] * d[..., 1]) + d[..., 2] * d[..., 2])

        old, new = length(a, b), length(a + dt * va, b + dt * vb)
        return (np.abs((new - len0) / len0) > 0.1) | (np.abs((new - old) / old) > 0.1)

    first = over(x[i], x[j], av[i], av[j], sc.bond_len0)
    todo = set(np.flatnonzero(first).tolist())
    done = last = 0
    for _ in range(max_sweeps):
        heap, again, last = sorted(todo), set(), 0
        queued = set(heap)
        while heap:
            e = heapq.heappop(heap)
            a, b = sc.bonds[e]
            if not over(x[a], x[b], av[a], av[b], sc.bond_len0[e]):
                continue
            av[a] = av[b] = 0.5 * (av[a] + av[b])
            last += 1
            again.add(e)
            for o in ((e - 1) % n, (e + 1) % n):  # the bonds that share a or b
                if o < e:
                    again.add(o)
                elif o > e and o not in queued:
                    queued.add(o)
                    heapq.heappush(heap, o)
        todo = again
        done += 1
        if last == 0:
            break
    return av, done, last


@pytest.mark.parametrize("n", [3, 64, 65, 1 << 20])
def test_closed_string_matches_the_sequential_sweeps(n):
    sc = closed_string(n)
    av, done, last = sweeps(sc)
    solver = solver_for_scene(sc, pass_timing=0)
    rep = solver.step()
    out = solver.getState()
    solver.close()
    assert (rep.status, rep.hit_pairs) == (0, 0)
    assert (rep.strain_sweeps, rep.strain_edges) == (done, last) and done >= 3
    assert np.array_equal(out["avg_vel"], av)
