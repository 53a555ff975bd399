"""The oracle's checking form (canonical order, deterministic functions) deals
its query and the search for pairs without a hit to all processors: the results
are those of one, and its pass counts and pair log are those of the serial form."""
import hashlib
import os
import subprocess
import sys

import numpy as np

from collision_amd import scenes as S
from oracle import oracle as O

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
STEPS = 24


def run(math_mode):
    sc = S.combined_scene(n=32, nstrings=6)
    o = O.OracleSolver(sc, log_pairs=1, order_mode=O.ORDER_CANONICAL, math_mode=math_mode)
    digest, told = hashlib.sha1(), []
    for _ in range(STEPS):
        rep = o.step()
        st = o.get_state()
        for k in sorted(st):
            digest.update(st[k].tobytes())
        digest.update(o.zone_labels().tobytes())
        told.append((rep.as_dict(), o.passes(), o.pair_log().tolist()))
    o.close()
    return digest.hexdigest(), told


def digest_with(threads):
    code = "from tests import test_oracle_threads as t; print(t.run(t.O.MATH_DET)[0])"
    return subprocess.run([sys.executable, "-c", code], cwd=ROOT, check=True, capture_output=True,
                          text=True, env=dict(os.environ, OMP_NUM_THREADS=str(threads))).stdout.strip()


def test_results_do_not_depend_on_the_processors():
    assert digest_with(1) == digest_with(3) == digest_with(8)


def test_checking_form_finds_what_the_serial_form_finds():
    (_, a), (_, b) = run(O.MATH_DET), run(O.MATH_LIBM)
    assert sum(r["hit_pairs"] for r, _, _ in a) > 0
    for (_, pa, la), (_, pb, lb) in zip(a, b):
        assert pa == pb and np.array_equal(la, lb)
