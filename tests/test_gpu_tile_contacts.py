"""Collision tiles at the edges of their contact phase: waves with more than 64
candidates near enough for the exact test, voxels with more than twelve
candidates and with more than a list holds, voxel counts at wave and workgroup
edges, several robots of a tile listing in the same step.  The tiled kernel equals
the plain one (a launch per phase and robot) bit for bit, as its contacts are
summed in the same order with the same arithmetic."""
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
@pytest.mark.parametrize("dims,squeeze", [((4, 4, 4), 0.9), ((5, 5, 5), 0.72), ((9, 7, 1), 0.6), ((6, 6, 5), 0.5), ((1, 1, 2), 0.7),
                                          ((8, 8, 3), 0.8)])
def test_squeezed_blocks_tiled_equals_plain(precision, dims, squeeze):
    n = int(np.prod(dims))
    prob = dict(configs.config0(), dims=dims, cells=np.ones(n, np.int8), phase=np.linspace(0, 1, n), enable_collision=1)
    models = [vx3mi.Model.from_problem(prob)] * 3
    out = []
    for mode in (vx3mi.MODE_PLAIN, vx3mi.MODE_TILED):
        b = vx3mi.Batch(models, precision)
        for r in range(3):  # each robot its own jitter, so that they list at different steps
            pos = b.state(r)["pos"]
            c = pos.mean(axis=0)
            b.set_state(r, pos=c + squeeze * (pos - c) + np.random.default_rng(r).normal(scale=3e-5 * r, size=pos.shape))
        b.record_contacts()
        b.step(1, mode=mode)
        first = b.contact_pairs()
        b.step(23, mode=mode)
        out.append((b.state(), first, b.contact_pairs(), b.voxel_flags(), b.link_flags(), b.diverged()))
        b.close()
    (sp, fp, pp, vp, lp, dp), (st, ft, pt, vt, lt, dt) = out
    if n > 8 and squeeze < 0.75:
        assert len(fp) > 0
    assert np.array_equal(fp, ft) and np.array_equal(dp, dt)
    for k in sp:
        assert np.array_equal(sp[k], st[k]), k
    assert np.array_equal(pp, pt) and np.array_equal(vp, vt)
    assert np.array_equal(lp[0], lt[0])
    stopped = np.repeat(dp != 0, models[0].nl)
    assert np.array_equal(lp[1][~stopped], lt[1][~stopped])  # strains of the running robots
    # a stopped robot's strains are formed again from what its last update left: one more rounding of the rest length
    np.testing.assert_allclose(lt[1][stopped], lp[1][stopped], rtol=4e-7 if precision == vx3mi.FP32 else 0)


@pytest.mark.parametrize("precision", [vx3mi.FP32, vx3mi.FP64])
@pytest.mark.parametrize("dims,E", [((4, 4, 4), 1e9), ((5, 5, 5), 3e8), ((9, 7, 1), 1e9), ((7, 5, 3), 3e8)])
def test_strains_of_stopped_robots_equal_the_plain_modes(precision, dims, E):
    """At a timestep too long for their moduli two of four robots pass the divergence
    strain inside a launch; the tiles form their links' strains again at its end."""
    n = int(np.prod(dims))
    base = configs.config0()
    models = [vx3mi.Model.from_problem(dict(base, dims=dims, cells=(np.arange(n) % 2 + 1).astype(np.int8), phase=np.linspace(0, 1, n),
                                            enable_collision=1, materials=[dict(configs.SOFT, E=e), dict(configs.SOFT, E=3 * e, cte=0.004)]))
              for e in (1e6, E, 1e6, 2 * E)]
    out = []
    for mode in (vx3mi.MODE_PLAIN, vx3mi.MODE_TILED):
        b = vx3mi.Batch(models, precision)
        for k in (1, 30, 40):
            b.step(k, dt=1e-5, mode=mode)
        out.append((b.diverged(), *b.link_flags(), b.state()["pos"]))
        b.close()
    assert out[0][0].tolist() == [0, 1, 0, 1]
    for plain, tiled in zip(*out):
        assert np.array_equal(plain, tiled)
