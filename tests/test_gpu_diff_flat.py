"""Differentiable steps as launches over the whole batch: a small robot gives the
same bits in a batch with a large one (flat steps) as alone (one workgroup per
robot), forward state and gradients, with the whole tape kept and with
checkpoints, at step counts on both sides of a checkpoint."""
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
@pytest.mark.parametrize("dims", [(1, 1, 1), (4, 3, 3), (5, 5, 3)])
@pytest.mark.parametrize("every,steps", [(0, 1), (0, 41), (13, 39), (13, 40), (40, 40)])
def test_flat_steps_equal_a_workgroup_per_robot(precision, dims, every, steps):
    small, large = configs.config3(seed=2, dims=dims), configs.config3(seed=3, dims=(11, 9, 9))
    ms, ml = vx3mi.Model.from_problem(small), vx3mi.Model.from_problem(large)
    assert ml.nl > 2 * 650 > 4 * ms.nl  # on either side of where the two ways cost the same
    out = []
    g = np.random.default_rng(1).normal(size=(ms.nv, 10))
    for models in ([ms], [ms, ml], [ml, ms]):
        d = vx3mi.Diff(models, precision, checkpoint_every=every)
        at = sum(m.nv for m in models[:models.index(ms)])
        d.forward(steps)
        s = d.state(models.index(ms))
        bars = []
        for a, b in ((0, 3), (3, 7), (7, 10)):
            full = np.zeros((d.nv, b - a))
            full[at:at + ms.nv] = g[:, a:b]
            bars.append(full)
        gp, ge = d.backward(grad_pos=bars[0], grad_quat=bars[1], grad_linmom=bars[2])
        out.append((s, gp[at:at + ms.nv], ge[at:at + ms.nv]))
        d.close()
    for s, gp, ge in out[1:]:
        for k in s:
            assert np.array_equal(s[k], out[0][0][k]), k
        np.testing.assert_array_equal(gp, out[0][1])
        np.testing.assert_array_equal(ge, out[0][2])


@pytest.mark.parametrize("precision", [vx3mi.FP32, vx3mi.FP64])
@pytest.mark.parametrize("dims", [(1, 1, 1), (4, 3, 3), (11, 9, 9)])
def test_set_moduli_equal_the_models_own(precision, dims):
    """The moduli of a model go through the host's constants, set ones through the
    device's: the same bits in states and gradients."""
    prob = configs.config3(seed=4, dims=dims)
    n = prob["cells"].size
    E = np.float32(10.0 ** np.random.default_rng(2).uniform(5, 8, size=n)).astype(np.float64)
    own = vx3mi.Model.from_problem(dict(prob, voxel_E=E))
    other = vx3mi.Model.from_problem(dict(prob, voxel_E=np.full(n, 3e6), phase=np.zeros(n)))
    out = []
    for m in (own, other):
        d = vx3mi.Diff([m, m], precision)
        if m is other:
            d.set_params(np.tile(prob["phase"][prob["cells"] > 0], 2), np.tile(E[prob["cells"] > 0], 2))
        d.forward(25)
        out.append((d.state(), *d.backward(grad_pos=np.ones((d.nv, 3)))))
        d.close()
    (sa, pa, ea), (sb, pb, eb) = out
    for k in sa:
        assert np.array_equal(sa[k], sb[k]), k
    np.testing.assert_array_equal(pa, pb)
    np.testing.assert_array_equal(ea, eb)


@pytest.mark.parametrize("precision", [vx3mi.FP32, vx3mi.FP64])
@pytest.mark.parametrize("dims,robots", [((4, 3, 3), 1), ((7, 6, 6), 1), ((7, 6, 6), 300), ((10, 9, 9), 2)])
@pytest.mark.parametrize("every", [0, 9])
def test_each_sweeps_own_choice_equals_the_given_ones(precision, dims, robots, every):
    """The forward and the reverse steps are laid out each as costs least (7x6x6 robots
    in FP32: forward by workgroup, reverse flat); given layouts of the reverse sweep
    and the default give the same bits, with the whole tape and with recomputation."""
    models = [vx3mi.Model.from_problem(configs.config3(seed=5, dims=dims))] * robots
    g = np.random.default_rng(3).normal(size=(robots * models[0].nv, 3))
    out = []
    for threads in (0, 512 if precision == vx3mi.FP32 else 256, -1):
        d = vx3mi.Diff(models, precision, checkpoint_every=every, reverse_threads=threads)
        d.forward(23)
        out.append((d.state(), *d.backward(grad_pos=g)))
        d.close()
    for s, gp, ge in out[1:]:
        for k in s:
            assert np.array_equal(s[k], out[0][0][k]), k
        np.testing.assert_array_equal(gp, out[0][1])
        np.testing.assert_array_equal(ge, out[0][2])
