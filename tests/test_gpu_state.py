"""cs_set_state is over when it returns, for small states (which go through
pinned host memory) as for large ones: the handle's stream starts no work
before the legacy default stream's, so work queued there first is over too."""
import numpy as np
import pytest
import torch

from collision_amd import scenes as S
from collision_amd.solver import solver_for_scene

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [4, 32, 232], ids=["small", "medium", "large"])  # 4 MB: 203 x 203
def test_set_state_has_ended_when_it_returns(n):
    sc = S.self_collision_cloth(n=n)
    solver = solver_for_scene(sc)
    x, vel = np.array(sc.x), np.array(sc.vel)
    solver.setState(x, vel)
    torch.cuda.synchronize()
    over = torch.cuda.Event()
    torch.cuda._sleep(50_000_000)  # tens of milliseconds on the default stream
    over.record()
    solver.setState(x + 1.0, vel)
    assert over.query()
    out = solver.getState()
    solver.close()
    assert np.array_equal(out["x"], x + 1.0) and np.array_equal(out["vel"], vel)
