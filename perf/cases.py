"""The collision step's workloads, as a program that uses this package runs them.

A simulation case is a mesh assembled once on a solver handle and a stretch of
time steps from a state of the running simulation: the program hands the
state over (setState), advances it (step / stepBatch: the predictor and
resolveCollision) and takes it back (getState).  The scenes are the generators
of `collision_amd.scenes` at the sizes of its configurations and around them;
every start state is one in which the scene's contacts are under way, reached
by free flight (`flight` steps, nothing but x += dt v) and by `warm` steps of
the solver.  The learned cases run the time-of-impact network on a batch of
CCD sub-test features.
"""
from __future__ import annotations

import math

import numpy as np
import torch

from collision_amd import scenes as S
from collision_amd.solver import CollisionSolver3d, solver_for_scene

H, IN, OUT = 128, 24, 2  # the network: 24 -> 128 -> 128 -> 2


def listed():
    return [
        # two crossing strings, 80 bonds: a few hundred microseconds a step, all of it latency
        dict(name="strings", kind="strings", n=40, flight=20, warm=4, steps=16, form="plain"),
        # a movable rigid ball rising into a falling slab: every pass walks the whole tree
        dict(name="bodies", kind="bodies", n=2, flight=40, warm=6, steps=8, form="plain"),
        # 32 x 32 cloth coming to rest on a sphere, with the captured step prologue
        dict(name="sheet32", kind="sheet", n=32, flight=240, warm=24, steps=8, form="graph"),
        # wavy cloths with random velocities: every edge over the strain limit, contacts everywhere
        dict(name="wavy64", kind="wavy", n=64, flight=0, warm=8, steps=4, form="plain"),
        dict(name="wavy256", kind="wavy", n=256, flight=0, warm=4, steps=2, form="plain"),
        # the same at an odd size, with the mixed-precision screens
        dict(name="wavy181_mixed", kind="wavy", n=181, flight=0, warm=4, steps=3, form="mixed"),
        # cloth over boxes under strings, many impact-zone passes a step: small, medium, the largest
        dict(name="drape96", kind="drape", n=96, flight=0, warm=32, steps=4, form="plain"),
        dict(name="drape256", kind="drape", n=256, flight=0, warm=28, steps=3, form="plain"),
        dict(name="drape1024", kind="drape", n=1024, flight=0, warm=24, steps=2, form="plain"),
        # 64 independent cloth-over-sphere scenes in one mesh
        dict(name="batch64", kind="batch", n=64, flight=140, warm=24, steps=2, form="plain"),
        # the time-of-impact network: scoring many sub-tests, and the gradient of one training batch
        dict(name="learned_infer", kind="infer", n=200003, form="plain"),
        dict(name="learned_grad", kind="grad", n=8192, form="plain"),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["strings", "bodies", "sheet", "wavy", "wavy", "drape", "drape", "batch", "infer", "grad"])
    if kind == "infer":
        return dict(kind=kind, n=_log_int(rng, 1, 400000), form="plain")
    if kind == "grad":
        return dict(kind=kind, n=_log_int(rng, 1, 20000), form="plain")
    form = rng.choice(["plain", "plain", "graph", "mixed", "learned"])
    if kind == "strings":
        n, flight, warm, steps = _log_int(rng, 5, 400), rng.randint(16, 22), rng.randint(1, 6), rng.randint(6, 20)
    elif kind == "bodies":
        n, flight, warm, steps = rng.randint(1, 3), rng.randint(36, 44), rng.randint(2, 10), rng.randint(4, 10)
    elif kind == "sheet":
        n, flight, warm, steps = _log_int(rng, 9, 128), rng.randint(236, 246), rng.randint(6, 24), rng.randint(3, 10)
    elif kind == "wavy":
        n, flight, warm, steps = _log_int(rng, 17, 300), 0, rng.randint(1, 8), rng.randint(1, 3)
    elif kind == "drape":
        n, flight, warm, steps = _log_int(rng, 41, 700), 0, rng.randint(18, 34), rng.randint(1, 2)
    else:
        n, flight, warm, steps = _log_int(rng, 2, 96), rng.randint(136, 142), rng.randint(4, 24), rng.randint(1, 3)
        form = rng.choice(["plain", "graph"])
    return dict(kind=kind, n=n, flight=flight, warm=warm, steps=steps, form=form)


def _scene(case, seed):
    kind, n = case["kind"], case["n"]
    if kind == "strings":
        return S.deck_string_string(segs=n)
    if kind == "bodies":
        return S.deck_ball_plane(level=n)
    if kind == "sheet":
        return S.cloth_over_sphere(n=n)
    if kind == "wavy":
        return S.self_collision_cloth(n=n, seed=S.seed_for(1) + seed)
    if kind == "drape":
        return S.combined_scene(n=n, nstrings=max(1, (n * n * 2000) >> 20))
    return S.batched_scenes(count=n, nmin=16, nmax=128, spacing=1.5)


def _weights(seed):
    g = np.random.default_rng(seed)
    w = []
    for rows, cols in ((H, IN), (H, H), (OUT, H)):
        lim = math.sqrt(6.0 / cols)
        w.append(g.uniform(-lim, lim, rows * cols))
        w.append(g.uniform(-0.1, 0.1, rows))
    return np.concatenate(w).astype(np.float32)


def _samples(case, seed):
    """sub-test features as the CCD pass forms them: four points within a few thicknesses of
    their centroid and their motion over the step, with labels"""
    g = np.random.default_rng(1000003 * seed + case["n"])
    x = g.normal(0.0, 2.0, (case["n"], IN))
    x[:, 12:] *= 0.5
    exists = (g.random(case["n"]) < 0.3).astype(np.float32)
    toi = (exists * g.random(case["n"])).astype(np.float32)
    return x.astype(np.float32), exists, toi


def prepare(case, seed):
    seed = int(seed)
    if case["kind"] in ("infer", "grad"):
        solver = CollisionSolver3d()
        solver.setLearnedWeights(_weights(5))
        x, exists, toi = _samples(case, seed)
        return dict(case=dict(case), solver=solver, x=x, exists=exists, toi=toi)
    sc = _scene(case, seed)
    # (passes are not timed in production; a batch is laid out wider than the default domain box)
    opts = dict(pass_timing=0, graph_step=int(case["form"] == "graph"),
                precision=int(case["form"] == "mixed"), learned=int(case["form"] == "learned"))
    if case["kind"] == "batch":
        opts.update(dom_lo=(-100.0,) * 3, dom_hi=(100.0,) * 3)
    solver = solver_for_scene(sc, **opts)
    if case["form"] == "learned":
        solver.setLearnedWeights(_weights(5))
    free = sc.fixed == 0
    if sc.vert_body is not None:
        free &= sc.vert_body < 0
    vel = sc.vel.copy()
    g = np.random.default_rng(seed)
    vel[free] += g.normal(0.0, 1e-3, (int(free.sum()), 3))
    x = sc.x + sc.vel * (sc.dt * case["flight"])
    solver.setState(x, vel)
    batch = case["kind"] == "batch"
    for _ in range(case["warm"]):
        solver.stepBatch() if batch else solver.step()
    at = solver.getState()
    return dict(case=dict(case), solver=solver, batch=batch, nbody=sc.nbody, x=at["x"], vel=at["vel"],
                has=at["has_collsn"])


def run(state):
    case, solver = state["case"], state["solver"]
    if case["kind"] == "infer":
        return solver.learnedInfer(state["x"])
    if case["kind"] == "grad":
        loss, grad = solver.learnedGrad(state["x"], state["exists"], state["toi"])
        return dict(loss=loss, grad=grad)
    solver.setState(state["x"], state["vel"], state["has"])
    told = []
    for _ in range(case["steps"]):
        if state["batch"]:
            rep, per = solver.stepBatch()
            told.append([r["n_passes"] for r in per] + [r["hit_pairs"] for r in per])
        else:
            rep = solver.step()
        told.append([rep.n_passes, rep.n_zones, rep.hit_pairs, rep.hit_subtests, rep.strain_sweeps])
    out = solver.getState()
    out["reports"] = np.concatenate([np.asarray(t, np.int64) for t in told])
    if state["nbody"]:
        out["com"], out["com_vel"] = solver.getBodies()
    return out


def work(case):
    n = case["n"]
    if case["kind"] == "infer":
        return dict(bytes=n * 4 * (IN + OUT), flops=2 * n * (IN * H + H * H + H * OUT))
    if case["kind"] == "grad":
        return dict(bytes=n * 4 * (IN + 2) + 4 * 19970 * 2, flops=6 * n * (IN * H + H * H + H * OUT) - 2 * n * IN * H)
    if case["kind"] == "strings":
        nv, nt, nb = 2 * (n + 1), 0, 2 * n
    elif case["kind"] == "bodies":
        nv, nt, nb = 10 + 10 * 4 ** n, 12 + 20 * 4 ** n, 0
    elif case["kind"] == "sheet":
        nv, nt, nb = n * n + 642, 2 * (n - 1) ** 2 + 1280, 0
    elif case["kind"] == "wavy":
        nv, nt, nb = n * n, 2 * (n - 1) ** 2, 0
    elif case["kind"] == "drape":
        m = max(1, (n * n * 2000) >> 20)
        nv, nt, nb = n * n + 32 + 65 * m, 2 * (n - 1) ** 2 + 48, 64 * m
    else:  # the mean cloth of a log-uniform side in [16, 128], and its sphere
        nv, nt, nb = n * (3880 + 402), n * (7600 + 800), 0
    # a step: state in (x, v) and out (x, v, x_old, the average velocity), the elements and their
    # rest lengths in; about one candidate pair an element, with its 15 proximity and 15 CCD
    # sub-tests of about 150 and 250 operations
    bytes_ = nv * (2 * 24 + 1 + 4 * 24 + 1) + nt * (12 + 4 + 24) + nb * (8 + 8)
    flops = 60 * nv + 15 * 400 * (nt + nb // 8)
    return dict(bytes=case["steps"] * bytes_, flops=case["steps"] * flops)


def _net(x, w):
    i = [0]

    def take(*shape):
        k = math.prod(shape)
        i[0] += k
        return w[i[0] - k:i[0]].reshape(shape)

    w1, b1, w2, b2, w3, b3 = (take(H, IN), take(H), take(H, H), take(H), take(OUT, H), take(OUT))
    return torch.relu(torch.relu(x @ w1.T + b1) @ w2.T + b2) @ w3.T + b3


def exact(case, seed):
    """The network and its training loss in 64 bits (from the FP32 weights, with no rounding of the
    activations).  The collision steps have no value of that kind: their impulses, zones and sweeps
    are defined by the order of their FP64 operations."""
    if case["kind"] not in ("infer", "grad"):
        return None
    x, exists, toi = _samples(case, int(seed))
    w = torch.tensor(_weights(5), dtype=torch.float64, requires_grad=case["kind"] == "grad")
    out = _net(torch.tensor(x, dtype=torch.float64), w)
    if case["kind"] == "infer":
        return out
    y, t = torch.tensor(exists, dtype=torch.float64), torch.tensor(toi, dtype=torch.float64)
    logit, seedv = out[:, 0], torch.sigmoid(out[:, 1])
    loss = (torch.nn.functional.softplus(logit) - logit * y + y * (seedv - t) ** 2).mean()
    loss.backward()
    return dict(loss=float(loss.detach()), grad=w.grad)
