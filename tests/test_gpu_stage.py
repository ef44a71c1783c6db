"""State read back through the pinned buffer: voxel counts at the edges of its
chunks (4,096 voxels of state, 5,461 of a frame), one robot of several, several
threads at once.  What comes back is what was set."""
import os
import sys
import threading

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path[:0] = [os.path.join(ROOT, "voxcraft-sim_amd")]

import vx3mi  # noqa: E402
from vx3mi import configs  # noqa: E402

pytestmark = pytest.mark.gpu


def random_state(n, seed):
    # values that FP32 holds exactly; positions are kept relative to the lattice there, so they stay whole lattice steps
    rng = np.random.default_rng(seed)
    whole = lambda *s: rng.integers(-1000, 1000, size=s).astype(np.float64)  # noqa: E731
    return dict(quat=whole(n, 4), linmom=whole(n, 3), angmom=whole(n, 3))


@pytest.mark.parametrize("precision", [vx3mi.FP32, vx3mi.FP64])
@pytest.mark.parametrize("counts", [(1,), (4095,), (4096,), (4097, 3), (1, 8193, 2), (5462, 10923)])
def test_state_comes_back_as_set(precision, counts):
    models = []
    for n in counts:
        prob = dict(configs.config0(), dims=(n if n < 1024 else 683, 1 if n < 1024 else -(-n // 683), 1))
        cells = np.zeros(int(np.prod(prob["dims"])), np.int8)
        cells[:n] = 1
        models.append(vx3mi.Model.from_problem(dict(prob, cells=cells, phase=np.zeros(cells.size), enable_collision=0)))
    b = vx3mi.Batch(models, precision)
    want = random_state(b.nv, 5)
    before = b.state()["pos"]
    b.set_state(-1, **want)
    got = b.state()
    assert np.array_equal(got["pos"], before)
    for k in want:
        assert np.array_equal(got[k], want[k]), k
    off = 0
    for r, n in enumerate(counts):
        s = b.state(r)
        for k in want:
            assert np.array_equal(s[k], want[k][off : off + n]), (r, k)
        off += n
    b.close()


def test_threads_read_at_once():
    prob = dict(configs.config0(), dims=(20, 20, 15), cells=np.ones(6000, np.int8), phase=np.zeros(6000), enable_collision=0)
    b = vx3mi.Batch([vx3mi.Model.from_problem(prob)], vx3mi.FP64)
    want = random_state(6000, 7)
    b.set_state(-1, **want)
    bad = []

    def read():
        for _ in range(10):
            s = b.state()
            bad.extend(k for k in want if not np.array_equal(s[k], want[k]))

    threads = [threading.Thread(target=read) for _ in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    b.close()
    assert not bad
