"""The mode of a batch that is not tuned, on both sides of where a tiled and a flat
step cost the same (each case 15 % or more from it), told by the launches of a call:
a tiled call of up to 1,000 steps is one."""
import os
import sys

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
