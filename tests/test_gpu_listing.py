"""Candidate lists at the edges of their making: more records around a voxel than
the queue of its lanes holds, more candidates than a list holds, voxel counts at
the edges of a lane group, wave and workgroup.  The flat and plain modes list with
a wave's lanes, the persistent mode with one lane a voxel; contacts, which are
summed in the lists' order, come out the same bit for bit."""
import os
import sys

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path[:0] = [os.path.join(ROOT, "voxcraft-sim_amd")]

import vx3mi  # noqa: E402
from vx3mi import configs  # noqa: E402

pytestmark = pytest.mark.gpu


def block_models(dims):
    n = int(np.prod(dims))
    prob = dict(configs.config0(), dims=dims, cells=np.ones(n, np.int8), phase=np.linspace(0, 1, n), enable_collision=1)
    return [vx3mi.Model.from_problem(prob)] * 3


def outcome(b):
    return dict(b.state(), pairs=b.contact_pairs(), flags=b.voxel_flags(), diverged=b.diverged())


def assert_same(a, b):
    for k in a:
        assert np.array_equal(a[k], b[k]), k


@pytest.mark.parametrize("precision", [vx3mi.FP32, vx3mi.FP64])
@pytest.mark.parametrize("dims,squeeze", [((1, 1, 2), 0.7), ((4, 4, 1), 0.6), ((5, 5, 5), 0.72), ((9, 7, 1), 0.5), ((6, 6, 5), 0.5),
                                          ((7, 6, 6), 0.3), ((12, 12, 12), 0.45)])
def test_lists_of_lanes_equal_lists_of_one_lane(precision, dims, squeeze):
    models = block_models(dims)
    out = []
    for mode in (vx3mi.MODE_PERSISTENT, vx3mi.MODE_FLAT, vx3mi.MODE_PLAIN):
        b = vx3mi.Batch(models, precision)
        for r in range(3):  # each robot its own jitter, so that they list at different steps
            pos = b.state(r)["pos"]
            c = pos.mean(axis=0)
            b.set_state(r, pos=c + squeeze * (pos - c) + np.random.default_rng(r).normal(scale=3e-5 * r, size=pos.shape))
        b.record_contacts()
        for _ in range(6):
            b.step(1, mode=mode)
        out.append(outcome(b))
        b.close()
    assert_same(out[0], out[1])
    assert_same(out[0], out[2])


@pytest.mark.parametrize("precision", [vx3mi.FP32, vx3mi.FP64])
@pytest.mark.parametrize("dims,squeeze,speed", [((4, 4, 4), 1.0, 0.0), ((5, 5, 5), 0.72, 0.0), ((7, 6, 6), 0.5, 0.0), ((9, 5, 3), 1.0, 3.0),
                                                ((6, 6, 5), 1.0, 30.0), ((20, 20, 12), 1.0, 3.0)])
def test_listings_beside_the_steps_equal_listings_before_them(precision, dims, squeeze, speed):
    """Calls of many flat steps start their listings some steps ahead; the plain
    mode lists before the step that needs it.  speed (m/s, falling apart towards
    the middle): voxels cross the skin of their lists within a few steps or one."""
    models = block_models(dims)
    out = []
    for mode in (vx3mi.MODE_PLAIN, vx3mi.MODE_FLAT):
        b = vx3mi.Batch(models, precision)
        for r in range(3):
            st = b.state(r)
            pos, c = st["pos"], st["pos"].mean(axis=0)
            mass = 1e6 * 0.01**3
            rng = np.random.default_rng(r)
            b.set_state(r, pos=c + squeeze * (pos - c) + rng.normal(scale=3e-5 * r, size=pos.shape),
                        linmom=speed * r * mass * rng.normal(size=pos.shape))
        b.record_contacts()
        for n in (1, 90, 7, 8, 33):  # listings before each step and beside them in turn
            b.step(n, mode=mode)
        out.append(outcome(b))
        listings = b.listings()
        b.close()
    assert_same(out[0], out[1])
    assert (listings > 0).all()


@pytest.mark.parametrize("precision", [vx3mi.FP32, vx3mi.FP64])
@pytest.mark.parametrize("var", ["t", "hit"])
def test_force_fields_of_long_calls_equal_the_plain_mode(precision, var):
    """Fields beside the contacts, and after them where they read the collision
    count: squeezed blocks of two materials, one of them a target, so that hits come."""
    n = 60
    base = configs.config0()
    soft = base["materials"][0]
    prob = dict(base, dims=(5, 4, 3), cells=(np.arange(n) % 2 + 1).astype(np.int8), phase=np.linspace(0, 1, n), enable_collision=1,
                materials=[soft, dict(soft, is_target=1)],
                force_field={"x": ("mtMUL", ("mtCONST", 1e-3), ("mtVAR", var)), "z": ("mtCONST", 1e-3)})
    models = [vx3mi.Model.from_problem(prob)] * 2 + block_models((4, 3, 3))[:1]
    out = []
    for mode in (vx3mi.MODE_PLAIN, vx3mi.MODE_FLAT):
        b = vx3mi.Batch(models, precision)
        pos = b.state(0)["pos"]
        c = pos.mean(axis=0)
        b.set_state(0, pos=c + 0.6 * (pos - c))
        for k in (3, 40):
            b.step(k, mode=mode)
        out.append(dict(b.state(), hits=b.hits()))
        b.close()
    assert out[0]["hits"][0] > 0
    assert_same(*out)


@pytest.mark.parametrize("precision", [vx3mi.FP32, vx3mi.FP64])
@pytest.mark.parametrize("calls", [[(vx3mi.MODE_FLAT, 8), (vx3mi.MODE_PERSISTENT, 1), (vx3mi.MODE_PERSISTENT, 8), (vx3mi.MODE_FLAT, 7)],
                                   [(vx3mi.MODE_TILED, 9), (vx3mi.MODE_PERSISTENT, 8), (vx3mi.MODE_FLAT, 20), (vx3mi.MODE_TILED, 7)]])
def test_modes_in_turn_equal_the_plain_mode(precision, calls):
    """Robots of different speeds whose lists are stale at the end of a call list
    in the first step of the next, whichever mode it takes."""
    models = block_models((7, 6, 6))
    out = []
    for plain in (True, False):
        b = vx3mi.Batch(models, precision)
        for r in range(3):
            pos = b.state(r)["pos"]
            c, rng = pos.mean(axis=0), np.random.default_rng(r)
            b.set_state(r, pos=c + 0.5 * (pos - c) + rng.normal(scale=3e-5 * r, size=pos.shape),
                        linmom=0.5 * r * rng.normal(size=pos.shape))
        for mode, n in calls:
            b.step(n, mode=vx3mi.MODE_PLAIN if plain else mode)
        out.append(dict(b.state(), flags=b.voxel_flags(), diverged=b.diverged()))
        b.close()
    assert_same(*out)


# per case: extents, speed of the whole robot and of each voxel by itself (m/s)
@pytest.mark.parametrize("precision", [vx3mi.FP32, vx3mi.FP64])
@pytest.mark.parametrize("dims,drift,jitter", [((4, 4, 4), 0.3, 0.0), ((9, 5, 3), 0.05, 0.3), ((5, 5, 5), 3.0, 0.0), ((7, 6, 6), 0.0, 3.0),
                                               ((14, 12, 8), 0.3, 0.0)])
def test_long_flat_calls_list_in_the_plain_modes_steps(precision, dims, drift, jitter):
    """Calls of many flat steps fill the grid of a listing in the voxel updates; the
    plain mode has a launch for it.  The same rule says when, so the listings of each
    robot are as many, and states and contacts the same bits."""
    models = block_models(dims)
    out = []
    for mode in (vx3mi.MODE_PLAIN, vx3mi.MODE_FLAT):
        b = vx3mi.Batch(models, precision)
        for r in range(3):
            rng = np.random.default_rng(r)
            v = np.full((models[r].nv, 3), drift * (r + 1)) + jitter * rng.normal(size=(models[r].nv, 3))
            b.set_state(r, linmom=1e-3 * v)  # a voxel weighs a gram
        counts = []
        for n in (60, 8, 1, 40):
            b.record_contacts()
            b.step(n, mode=mode)
            counts.append(b.listings())
        out.append(dict(outcome(b), counts=np.array(counts)))
        b.close()
    assert_same(*out)
    assert (out[0]["counts"][-1] > 2).all()


@pytest.mark.parametrize("precision", [vx3mi.FP32, vx3mi.FP64])
@pytest.mark.parametrize("speed", [0.0, 0.5, 4.0])
def test_large_bodies_in_long_flat_calls_equal_the_plain_mode(precision, speed):
    """A body of more than two count workgroups' surface voxels, at rest and thrown."""
    model = vx3mi.Model.from_problem(configs.config1(seed=2, dims=(40, 40, 8)))
    assert model.ns > 2 * 4096
    out = []
    for mode in (vx3mi.MODE_PLAIN, vx3mi.MODE_FLAT):
        b = vx3mi.Batch([model], precision)
        b.set_state(0, linmom=np.full((model.nv, 3), speed * 1e-3))
        b.record_contacts()
        for n in (75, 30):
            b.step(n, mode=mode)
        out.append(dict(outcome(b), listings=b.listings()))
        b.close()
    assert_same(*out)


@pytest.mark.parametrize("precision", [vx3mi.FP32, vx3mi.FP64])
def test_many_materials_in_long_flat_calls_equal_the_plain_mode(precision):
    """More voxel materials than the contact phase keeps the sizes of (64)."""
    base = configs.config0()
    models = []
    for k in range(40):
        mats = [dict(base["materials"][0], E=1e6 * (1 + 0.01 * k)), dict(base["materials"][0], E=2e6 * (1 + 0.01 * k))]
        models.append(vx3mi.Model.from_problem(dict(base, dims=(4, 3, 3), cells=(np.arange(36) % 2 + 1).astype(np.int8),
                                                    phase=np.linspace(0, 1, 36), materials=mats, enable_collision=1)))
    out = []
    for mode in (vx3mi.MODE_PLAIN, vx3mi.MODE_FLAT):
        b = vx3mi.Batch(models, precision)
        for r in range(40):
            pos = b.state(r)["pos"]
            c = pos.mean(axis=0)
            b.set_state(r, pos=c + (0.6 + 0.01 * r) * (pos - c))
        b.record_contacts()
        b.step(1, mode=mode)
        first = b.contact_pairs()
        b.step(40, mode=mode)
        out.append(dict(outcome(b), first=first, listings=b.listings()))
        b.close()
    assert len(out[0]["first"]) > 0
    assert_same(*out)


@pytest.mark.parametrize("precision", [vx3mi.FP32, vx3mi.FP64])
def test_a_blow_in_a_long_flat_call_equals_the_plain_mode(precision):
    """Robots at rest that a force field throws within one step past the limit of
    their lists: no grid has been filled for the step after, which tests all pairs.
    A second robot is squeezed and has contacts meanwhile."""
    n = 5 * 4 * 4
    base = dict(configs.config0(), dims=(5, 4, 4), cells=np.ones(n, np.int8), phase=np.zeros(n), enable_collision=1, vary_temp=0,
                grav_acc=0.0, floor_enabled=0, materials=[dict(configs.SOFT, cte=0.0)])
    dt = vx3mi.Model.from_problem(base).recommended_dt() * base["dt_frac"]
    limit = 0.49 * 0.15 * 0.01
    force = 3 * limit * 1e-3 / dt**2  # on a gram
    prob = dict(base, force_field={"x": ("mtMUL", ("mtCONST", force), ("mtGREATERTHAN", ("mtVAR", "t"), ("mtCONST", 20.5 * dt)))})
    models = [vx3mi.Model.from_problem(prob)] * 2
    trace = []
    out = []
    for mode in (vx3mi.MODE_PLAIN, vx3mi.MODE_FLAT):
        b = vx3mi.Batch(models, precision)
        pos = b.state(1)["pos"]
        c = pos.mean(axis=0)
        b.set_state(1, pos=c + 0.97 * (pos - c))
        b.record_contacts()
        if mode == vx3mi.MODE_PLAIN:
            for _ in range(40):
                b.step(1, mode=mode)
                trace.append(b.state(0)["pos"])
        else:
            b.step(40, mode=mode)
        out.append(dict(b.state(), flags=b.voxel_flags(), diverged=b.diverged()))
        b.close()
    step = np.array([np.abs(y - x).max() for x, y in zip(trace, trace[1:])])
    k = int(np.argmax(step > limit))
    assert k > 10 and step[:k].max() < 0.1 * limit and step[k] > limit  # from rest past the limit in one step
    assert_same(*out)


@pytest.mark.parametrize("precision", [vx3mi.FP32, vx3mi.FP64])
def test_a_fast_bodys_steps_cost_a_listing_at_the_most(precision):
    """A thrown body of 8,222 surface voxels lists in every step.  A listing costs
    about a step; a step that tests all their pairs costs more than fifty."""
    model = vx3mi.Model.from_problem(dict(configs.config1(seed=2, dims=(40, 40, 8)), slow_damp_z=0.0))
    us = []
    for speed in (0.0, 200.0):
        b = vx3mi.Batch([model], precision)
        b.step(40, mode=vx3mi.MODE_FLAT)
        b.set_state(0, linmom=np.tile([0, 0, speed * 1e-3], (model.nv, 1)))
        b.step(10, mode=vx3mi.MODE_FLAT)
        before = b.listings()[0]
        b.step(60, mode=vx3mi.MODE_FLAT)
        us.append(b.last_step_ms() * 1e3 / 60)
        listed = b.listings()[0] - before
        b.close()
    assert listed > 40
    assert us[1] < 8 * us[0], us


@pytest.mark.parametrize("precision", [vx3mi.FP32, vx3mi.FP64])
@pytest.mark.parametrize("far", [60, 700, 1000])
def test_contacts_between_distant_lattice_sites_equal_the_plain_mode(precision, far):
    """Two blocks of one robot, far apart in the lattice and put side by side at
    distances around the contact envelope: their FP32 positions are kept relative to
    their sites, hundreds of lattice lengths away, where rounding is a fair part of
    what the first test of a candidate rounds its radius up by."""
    dims = (far + 3, 3, 3)
    cells = np.zeros(dims[::-1], np.int8)
    cells[:, :, :3] = cells[:, :, far:] = 1
    prob = dict(configs.config0(), dims=dims, cells=cells.reshape(-1), phase=np.linspace(0, 1, 54), enable_collision=1, grav_acc=0.0,
                floor_enabled=0, materials=[dict(configs.SOFT, cte=0.0)])
    models = [vx3mi.Model.from_problem(prob)] * 24
    out = []
    for mode in (vx3mi.MODE_PLAIN, vx3mi.MODE_FLAT):
        b = vx3mi.Batch(models, precision)
        for r in range(24):
            pos = b.state(r)["pos"]
            other = pos[:, 0] > 0.01 * (far - 0.5)
            pos[other, 0] -= 0.01 * far
            pos[other, 1] += 0.01 * (2 + 1.25 * (1 + (r - 12) * 4e-6))  # the envelope is 1.25 voxels
            b.set_state(r, pos=pos)
        b.record_contacts()
        pairs = []
        for n in (1, 9, 30):
            b.step(n, mode=mode)
            pairs.append(b.contact_pairs())
        out.append(dict(outcome(b), first=pairs[0], then=pairs[1]))
        b.close()
    assert 0 < len(out[0]["first"])
    assert_same(*out)
