"""The mode of a batch that is not tuned, on both sides of where a tiled and a flat
step cost the same (each case 15 % or more from it), told by the launches of a call:
a tiled call of up to 1,000 steps is one."""
import os
import sys

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path[:0] = [os.path.join(ROOT, "voxcraft-sim_amd")]

import vx3mi  # noqa: E402
from vx3mi import configs  # noqa: E402

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision,collisions,robots,size,tiled", [
    (vx3mi.FP32, 1, 1, 11, False), (vx3mi.FP32, 1, 4, 11, False), (vx3mi.FP32, 1, 64, 11, True), (vx3mi.FP32, 1, 1, 8, True),
    (vx3mi.FP32, 0, 1, 11, True), (vx3mi.FP32, 0, 600, 10, True),
    (vx3mi.FP64, 0, 1, 6, True), (vx3mi.FP64, 0, 1500, 8, True),  # three rounds of tiles
    (vx3mi.FP64, 1, 1, 6, True), (vx3mi.FP64, 1, 400, 8, True), (vx3mi.FP64, 1, 40, 11, False)])  # the last: no tile holds them
def test_default_mode(precision, collisions, robots, size, tiled):
    probs = configs.config2(seed=3, n=min(robots, 8), lo=size, hi=size, collisions=collisions)
    models = [vx3mi.Model.from_problem(p) for p in probs]
    b = vx3mi.Batch([models[r % len(models)] for r in range(robots)], precision)
    b.step(20)
    assert (b.last_step_launches() == 1) == tiled
    b.close()


@pytest.mark.parametrize("precision,robots", [(vx3mi.FP32, 128), (vx3mi.FP32, 32769), (vx3mi.FP64, 16385)])
def test_tiles_full_of_robots(precision, robots):
    """Robots so small that the tiles' robot count fills them, one more than a round
    of the device holds: each robot as alone, whatever tile it went to."""
    prob = dict(configs.config0(), dims=(2, 1, 1), cells=np.ones(2, np.int8))
    models = [vx3mi.Model.from_problem(dict(prob, phase=np.full(2, k / 7))) for k in range(7)]
    b = vx3mi.Batch([models[r % 7] for r in range(robots)], precision)
    b.step(40, mode=vx3mi.MODE_TILED)
    pos = b.state()["pos"].reshape(robots, 2, 3)
    b.close()
    for k in range(7):
        a = vx3mi.Batch([models[k]], precision)
        a.step(40, mode=vx3mi.MODE_FLAT)
        assert np.array_equal(pos[k::7], np.broadcast_to(a.state()["pos"], pos[k::7].shape))
        a.close()
