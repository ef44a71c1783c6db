"""Flat steps that run as captured graphs of 1000 and 64 steps: batches that no
other form of the flat mode takes (no collisions, or robots that lose voxels), in
one call, in calls that start at odd steps and in single steps.  The same bits."""
import os
import sys

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path[:0] = [os.path.join(ROOT, "voxcraft-sim_amd")]

import vx3mi  # noqa: E402
from vx3mi import configs  # noqa: E402

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", [vx3mi.FP32, vx3mi.FP64])
@pytest.mark.parametrize("collisions", [0, 1])
def test_graph_chunks_equal_single_steps(precision, collisions):
    probs = configs.config2(seed=5, n=6, hi=8, collisions=collisions)
    if collisions:  # voxels leave some hundred steps into the run
        dt = vx3mi.Model.from_problem(probs[0]).recommended_dt() * probs[0]["dt_frac"]
        probs = [dict(p, secondary_experiment=1, materials=[configs.SOFT, dict(configs.STIFF, remove_after=(300.5 + 500 * r) * dt)])
                 for r, p in enumerate(probs)]
    models = [vx3mi.Model.from_problem(p) for p in probs]
    out = []
    for calls in ([2130], [63] + [64] * 32 + [19], [1] * 2130):
        b = vx3mi.Batch(models, precision)
        b.step(1, mode=vx3mi.MODE_FLAT)
        launches = b.last_step_launches()
        for n in calls:
            b.step(n, mode=vx3mi.MODE_FLAT)
            assert b.last_step_launches() == launches * n  # none around the steps: these are the captured ones
        out.append(dict(b.state(), time=b.time(), removed=b.removed()[0]))
        b.close()
    assert not collisions or (out[0]["removed"] > 0).any()
    for o in out[1:]:
        for k in o:
            assert np.array_equal(o[k], out[0][k]), k
