"""Inference of the proposer at the edges of its 16-sample tiles and of its
rounds (3,072 wavefronts of 16 samples fit the card at once).

Tolerance: the hidden activations are rounded to BF16 on both sides; sums in
another order (FP32 here, FP64 in the CPU network) can move single activations
by one BF16 step, 2^-8 of their value, and a few such steps among the 128 of
a layer stay below 1e-2 of the largest output of 1,000 such samples."""
import numpy as np
import pytest

from collision_amd.solver import CollisionSolver3d
from oracle import mlp as M

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 15, 16, 17, 63, 65, 49151, 49152, 49153, 98305])
def test_inference_matches_the_cpu_network(n):
    g = CollisionSolver3d()
    g.learnedInit(5)
    w = g.learnedWeights()
    x = np.random.default_rng(n).normal(0, 3, (n, 24)).astype(np.float32)
    out = g.learnedInfer(x)
    assert out.shape == (n, 2) and np.isfinite(out).all()
    rows = np.unique(np.concatenate([np.arange(min(n, 200)), np.arange(max(0, n - 200), n)]))
    ref = M.forward(w, x[rows], emulate_bf16=True)
    scale = np.abs(M.forward(w, np.random.default_rng(0).normal(0, 3, (1000, 24)),
                             emulate_bf16=True)).max()
    assert np.abs(out[rows] - ref).max() < 1e-2 * scale
    # a row's outputs do not depend on its place
    np.testing.assert_array_equal(g.learnedInfer(x[n - 1:]), out[n - 1:])
    g.close()
