"""The work a user of this framework has it do, as cases to be timed.

A case is one of four kinds, each a pass through the public entry points:

* ``step``  -- a batch of robots advanced some timesteps, then its state read
  (``Batch.step`` / ``Batch.state``): a control loop, a design study, a population
  under evolution, one large body; in both precisions, collisions on and off.
* ``run``   -- the simulation driver with its report and ``.history`` text
  (``vx3mi.run``), the drop-in for the reference's executable, in its precision.
* ``diff``  -- the differentiable timestep forward and backward through
  ``torch_diff.simulate``: gradients of a travelled distance with respect to each
  voxel's actuation phase and stiffness.

``exact`` integrates the same robots in float64 with plain torch (forward
equations below; gradients by autograd, one step at a time).
"""
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "voxcraft-sim_amd"))

import vx3mi  # noqa: E402
from vx3mi import configs, torch_diff  # noqa: E402
from vx3mi import vxa as vxa_text  # noqa: E402


def listed():
    return [
        # a controller that looks at a 4x4x4 robot every ten steps: the smallest call, latency only
        dict(name="control_loop_fp64", kind="step", shape=1, bits=64, robots=1, lo=4, hi=4, fill=1.0, collide=0, extras=0, steps=10),
        # one demo-sized robot watched while it moves, single precision, collisions on (the default)
        dict(name="robot_fp32", kind="step", shape=2, bits=32, robots=1, lo=8, hi=8, fill=0.8, collide=1, extras=0, steps=301),
        # the same in the reference's precision, a smaller uneven body
        dict(name="robot_fp64", kind="step", shape=3, bits=64, robots=1, lo=5, hi=8, fill=0.7, collide=1, extras=0, steps=333),
        # one large body with collisions (64 x 64 x 16 cells, 45,800 voxels)
        dict(name="body_fp32", kind="step", shape=4, bits=32, robots=1, lo=64, hi=64, flat=16, fill=0.7, collide=1, extras=0, steps=500),
        # a large body in the reference's precision, odd extents
        dict(name="body_fp64", kind="step", shape=5, bits=64, robots=1, lo=37, hi=45, flat=13, fill=0.7, collide=1, extras=0, steps=150),
        # a population under evolution, one generation's chunk: 1024 uneven robots, collisions off
        dict(name="population_fp32", kind="step", shape=6, bits=32, robots=1024, lo=4, hi=12, fill=0.6, collide=0, extras=0, steps=1000),
        # the same with collisions on
        dict(name="population_collide_fp32", kind="step", shape=7, bits=32, robots=1024, lo=4, hi=12, fill=0.6, collide=1, extras=0, steps=300),
        # a smaller population in the reference's precision, collisions on
        dict(name="population_collide_fp64", kind="step", shape=8, bits=64, robots=200, lo=4, hi=12, fill=0.6, collide=1, extras=0, steps=200),
        # robots with signals, cilia and force fields
        dict(name="extras_fp32", kind="step", shape=9, bits=32, robots=48, lo=5, hi=9, fill=0.8, collide=1, extras=1, steps=300),
        # the simulation driver: report, history frames, fitness
        dict(name="driver_history_fp64", kind="run", shape=10, bits=64, robots=8, lo=4, hi=7, fill=0.8, collide=1, steps=600),
        # gradient of one 8x8x8 robot's travel (co-design of phase and stiffness)
        dict(name="gradient_fp32", kind="diff", shape=11, bits=32, robots=1, lo=8, hi=8, fill=1.0, steps=400),
        # gradients of a batch of uneven robots
        dict(name="gradient_population_fp32", kind="diff", shape=12, bits=32, robots=128, lo=6, hi=16, fill=0.6, steps=150),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case of the ranges above (shape: which bodies; their actuation and stiffness are the inputs)."""
    shape = rng.randrange(100, 1 << 20)
    what = rng.choice(["robot", "robot", "body", "population", "population", "extras", "run", "diff", "diff"])
    if what == "robot":
        lo = rng.randint(3, 9)
        return dict(kind="step", shape=shape, bits=rng.choice([32, 64]), robots=1, lo=lo, hi=lo + rng.randint(0, 3),
                    fill=round(rng.uniform(0.55, 1.0), 3), collide=rng.randint(0, 1), extras=0, steps=_log(rng, 7, 900))
    if what == "body":
        lo = _log(rng, 14, 50)
        return dict(kind="step", shape=shape, bits=rng.choice([32, 32, 64]), robots=1, lo=lo, hi=lo + rng.randint(0, 12),
                    flat=rng.randint(6, 16), fill=round(rng.uniform(0.55, 0.9), 3), collide=rng.randint(0, 1), extras=0,
                    steps=_log(rng, 20, 200))
    if what == "population":
        bits = rng.choice([32, 32, 64])
        lo = rng.randint(3, 7)
        return dict(kind="step", shape=shape, bits=bits, robots=_log(rng, 3, 900 if bits == 32 else 150), lo=lo,
                    hi=rng.randint(lo, 12), fill=round(rng.uniform(0.55, 0.9), 3), collide=rng.randint(0, 1), extras=0,
                    steps=_log(rng, 30, 300))
    if what == "extras":
        lo = rng.randint(4, 6)
        return dict(kind="step", shape=shape, bits=rng.choice([32, 64]), robots=_log(rng, 2, 48), lo=lo, hi=rng.randint(lo, 9),
                    fill=round(rng.uniform(0.6, 0.95), 3), collide=1, extras=1, steps=_log(rng, 30, 300))
    if what == "run":
        lo = rng.randint(3, 6)
        return dict(kind="run", shape=shape, bits=64, robots=_log(rng, 1, 12), lo=lo, hi=rng.randint(lo, 8),
                    fill=round(rng.uniform(0.6, 1.0), 3), collide=rng.randint(0, 1), steps=_log(rng, 100, 600))
    if rng.random() < 0.5:
        lo = rng.randint(3, 9)
        return dict(kind="diff", shape=shape, bits=rng.choice([32, 32, 64]), robots=1, lo=lo, hi=lo + rng.randint(0, 2),
                    fill=round(rng.uniform(0.6, 1.0), 3), steps=_log(rng, 40, 400))
    lo = rng.randint(4, 8)
    return dict(kind="diff", shape=shape, bits=32, robots=_log(rng, 4, 120), lo=lo, hi=rng.randint(lo, 15),
                fill=round(rng.uniform(0.55, 0.8), 3), steps=_log(rng, 30, 150))


# ---- inputs ---------------------------------------------------------------------
def _problems(case, seed):
    """The robots of a case (cells and two materials, from its shape), and from the seed a random
    actuation phase per voxel (and stiffness, or cilia forces)."""
    body, rng = np.random.default_rng(case["shape"]), np.random.default_rng(seed)
    out = []
    for _ in range(case["robots"]):
        dims = body.integers(case["lo"], case["hi"] + 1, size=3)
        if case.get("flat"):
            dims[2] = case["flat"]
        grad = case["kind"] == "diff"
        p = configs.random_robot(body, dims, case["fill"] if case["fill"] < 1 else 2.0, two_materials=not grad,
                                 enable_collision=0 if grad else case["collide"])
        nv = int((p["cells"] > 0).sum())
        p["phase"] = rng.uniform(0.0, 1.0, size=nv)
        if grad:
            p["voxel_E"] = (10.0 ** rng.uniform(6.0, 7.0, size=nv)).astype(np.float32)
        if case.get("extras"):
            # pacemakers of the stiff material drive cilia; a weak force field along x
            sig = dict(signal_decay=0.85, signal_delay=0.0015, inactive_period=0.002, cilia=1.0)
            p["materials"] = [dict(configs.SOFT, **sig), dict(configs.STIFF, is_pacemaker=1, pacemaker_period=0.004, **sig)]
            p.update(enable_signals=1, enable_cilia=1, cilia_base=rng.normal(size=(nv, 3)) * 1e-4,
                     cilia_shift=rng.normal(size=(nv, 3)) * 2e-5,
                     force_field={"x": ("mtMUL", ("mtCONST", 1e-4), ("mtSIN", ("mtMUL", ("mtCONST", 60.0), ("mtVAR", "t"))))})
        out.append(p)
    return out


def prepare(case, seed):
    problems = _problems(case, seed)
    fp = vx3mi.FP32 if case["bits"] == 32 else vx3mi.FP64
    s = dict(case=case)
    if case["kind"] == "diff":
        models = [vx3mi.Model.from_problem(p) for p in problems]
        s["diff"] = vx3mi.Diff(models, fp)
        kind = torch.float32 if case["bits"] == 32 else torch.float64
        phase = np.concatenate([p["phase"] for p in problems])
        logE = np.log10(np.concatenate([p["voxel_E"] for p in problems]).astype(np.float64))
        s["psi"] = torch.tensor(phase * 2 * math.pi, dtype=kind)
        s["logE"] = torch.tensor(logE, dtype=kind)
        # the mean displacement along -x of each robot, summed
        s["weight"] = torch.tensor(np.concatenate([np.full(len(p["phase"]), -1.0 / len(p["phase"])) for p in problems]))
    elif case["kind"] == "run":
        s["models"] = [vx3mi.Model.from_xml(vxa_text.write_vxa(p, fitness=("mtVAR", "x"), record=(20, 1, 1))) for p in problems]
        s["batch"] = vx3mi.Batch(s["models"], fp)
        # at most one frame every 20 / (10000 dt) steps, 160 characters a voxel and 100 a link
        s["room"] = sum(1000 + (2 + case["steps"] // int(1 + 20 / (9000 * m.recommended_dt()))) * (200 + 160 * m.nv + 100 * m.nl)
                        for m in s["models"])
    else:
        s["batch"] = vx3mi.Batch([vx3mi.Model.from_problem(p) for p in problems], fp)
    return s


def _text(text, room):
    """The history's bytes in a buffer of a fixed size."""
    out = np.zeros(room, dtype=np.uint8)
    out[:len(text)] = np.frombuffer(text.encode(), dtype=np.uint8)
    return out


def run(state):
    case = state["case"]
    if case["kind"] == "diff":
        psi = state["psi"].clone().requires_grad_(True)
        logE = state["logE"].clone().requires_grad_(True)
        pos = torch_diff.simulate(state["diff"], psi / (2 * math.pi), 10.0 ** logE, case["steps"])
        (pos[:, 0] * state["weight"]).sum().backward()
        return dict(pos=pos.detach().to(psi.dtype), psi=psi.grad, logE=logE.grad)
    if case["kind"] == "run":
        results, history, final = vx3mi.run(state["batch"], state["models"], max_steps=case["steps"])
        return dict(pos=np.concatenate(final), fitness=np.array([r["fitness_score"] for r in results]),
                    com=np.array([r["current_com"] for r in results]), steps=np.array([r["steps"] for r in results]),
                    history=_text("".join(history), state["room"]))
    batch = state["batch"]
    batch.step(case["steps"])
    got = batch.state()
    if case["bits"] == 32:  # the state's own precision
        got = {k: v.astype(np.float32) for k, v in got.items()}
    return got


def work(case):
    """Each state read and written once in a pass; the arithmetic of its steps
    (about 450 operations a link, 320 a voxel and step; the adjoint about three
    times its forward)."""
    cells = case["robots"] * ((case["lo"] + case["hi"]) / 2) ** 3
    if case.get("flat"):
        cells = case["robots"] * ((case["lo"] + case["hi"]) / 2) ** 2 * case["flat"]
    v = cells * case["fill"]
    links = 3 * cells * case["fill"] ** 2
    real = case["bits"] / 8
    flops = case["steps"] * (320 * v + 450 * links)
    if case["kind"] == "diff":
        return dict(bytes=real * (v * 10 + links * 20), flops=4 * flops)
    return dict(bytes=2 * real * (v * 14 + links * 11), flops=flops)


# ---- the same robots in float64, by plain torch ------------------------------------
_DEV = "cuda" if torch.cuda.is_available() else "cpu"


def _qmul(a, b):
    aw, ax, ay, az = a.unbind(-1)
    bw, bx, by, bz = b.unbind(-1)
    return torch.stack([aw * bw - ax * bx - ay * by - az * bz, aw * bx + ax * bw + ay * bz - az * by,
                        aw * by - ax * bz + ay * bw + az * bx, aw * bz + ax * by - ay * bx + az * bw], -1)


def _conj(q):
    return torch.cat([q[..., :1], -q[..., 1:]], -1)


def _rot(q, f):
    w, v = q[..., :1], q[..., 1:]
    t = 2 * torch.linalg.cross(v, f)
    return f * (w * w + (v * v).sum(-1, keepdim=True)) + w * t + torch.linalg.cross(v, t)


def _rotvec(q):
    w, v = q[..., 0], q[..., 1:]
    s2 = (v * v).sum(-1)
    near = s2 < 2.4e-3
    s = torch.where(near, torch.ones_like(s2), s2).sqrt()
    k = torch.where(near, 2 * (2 / (1 + w)).sqrt(), 2 * torch.atan2(s, w) / s)
    return v * k[..., None]


def _from_rotvec(r):
    h = r / 2
    m2 = (h * h).sum(-1)
    tiny = m2 < 1e-6
    m = torch.where(tiny, torch.ones_like(m2), m2).sqrt()
    c = torch.where(tiny, 1 - m2 / 2 + m2 * m2 / 24, torch.cos(m))
    s = torch.where(tiny, 1 - m2 / 6 + m2 * m2 / 120, torch.sin(m) / m)
    return torch.cat([c[..., None], h * s[..., None]], -1)


def _to_x(d):
    """The rotation that takes the direction d onto +x (first order below 1.732e-2)."""
    y, z = d[..., 1] / d[..., 0], d[..., 2] / d[..., 0]
    near = (y.abs() < 1.732e-2) & (z.abs() < 1.732e-2)
    rho2 = d[..., 1] ** 2 + d[..., 2] ** 2
    rho = torch.where(near, torch.ones_like(rho2), rho2).sqrt()
    half = torch.atan2(rho, d[..., 0]) / 2
    far = torch.stack([torch.cos(half), torch.zeros_like(half), d[..., 2] / rho * torch.sin(half),
                       -d[..., 1] / rho * torch.sin(half)], -1)
    qy, qz = z / 2, -y / 2
    low = torch.stack([1 - (qy * qy + qz * qz) / 2, torch.zeros_like(qy), qy, qz], -1)
    return torch.where(near[..., None], low, far)


class _Body:
    """The robots of a case as tensors: lattice sites, links, materials, dt."""

    def __init__(self, problems, E=None, phase=None, diff=False):
        site, Ev, ph, rob, neg, pos, axis, dts, rho, first = [], [], [], [], [], [], [], [], [], 0
        p0 = problems[0]
        self.L = L = p0["lattice_dim"]
        self.diff = diff
        for r, p in enumerate(problems):
            nx, ny, nz = (int(n) for n in p["dims"])
            cells = np.asarray(p["cells"]).reshape(nz, ny, nx)
            zyx = np.argwhere(cells > 0)
            index = -np.ones(cells.shape, dtype=np.int64)
            index[cells > 0] = np.arange(len(zyx))
            mat = cells[cells > 0].astype(int) - 1
            Er = np.array([m["E"] for m in p["materials"]], dtype=np.float64)[mat]
            if p.get("voxel_E") is not None:
                Er = np.asarray(p["voxel_E"], dtype=np.float64)
            stiff = 0.0
            for ax, (lo, hi) in enumerate([(index[:, :, :-1], index[:, :, 1:]), (index[:, :-1], index[:, 1:]), (index[:-1], index[1:])]):
                both = (lo >= 0) & (hi >= 0)
                a, b = lo[both], hi[both]
                neg.append(a + first), pos.append(b + first), axis.append(np.full(len(a), ax))
                if len(a):
                    stiff = max(stiff, float((2 * Er[a] * Er[b] / (Er[a] + Er[b])).max()))
            stiff = 1e7 if diff else (stiff or float(Er.max()))
            mass = p["materials"][0]["rho"] * L ** 3
            dts.append(float(np.float32(p["dt_frac"] / (float(np.float32(6.283185)) * math.sqrt(stiff * L / mass)))))
            site.append(zyx[:, ::-1]), Ev.append(Er), ph.append(p["phase"]), rob.append(np.full(len(zyx), r))
            first += len(zyx)
        t = lambda a, k=torch.float64: torch.tensor(np.concatenate(a), dtype=k, device=_DEV)  # noqa: E731
        m = p0["materials"][0]
        self.site, self.rob = t(site), t(rob, torch.int64)
        self.neg, self.pos, self.axis = t(neg, torch.int64), t(pos, torch.int64), t(axis, torch.int64)
        self.E = t(Ev) if E is None else E
        self.phase = t(ph) if phase is None else phase
        if diff:
            dts = [min(dts)] * len(dts)
        self.dt = torch.tensor(dts, dtype=torch.float64, device=_DEV)[self.rob][:, None]
        self.dtl = self.dt[self.neg]
        self.mass, self.alpha = m["rho"] * L ** 3, m["cte"]
        self.inertia = self.mass * L * L / 6
        self.mu_s, self.mu_k = m["mu_s"], m["mu_k"]
        self.zi, self.zc, self.zg = p0["bond_damp_z"], p0["col_damp_z"], p0["slow_damp_z"]
        self.grav = self.mass * p0["grav_acc"]
        self.amp, self.period = p0["temp_amplitude"], p0["temp_period"]
        # toAxisX / back as index and sign per axis
        perm = torch.tensor([[0, 1, 2], [1, 0, 2], [2, 1, 0]], device=_DEV)
        sign = torch.tensor([[1, 1, 1], [1, -1, 1], [1, 1, -1]], dtype=torch.float64, device=_DEV)
        self.perm, self.sx = perm[self.axis], sign[self.axis]
        back = torch.tensor([[1, 1, 1], [-1, 1, 1], [-1, 1, 1]], dtype=torch.float64, device=_DEV)
        self.sb = back[self.axis]
        self.collide = bool(p0["enable_collision"]) and not diff
        if self.collide:
            links = torch.zeros(first, dtype=torch.int64, device=_DEV)
            one = torch.ones_like(self.neg)
            links.index_add_(0, self.neg, one), links.index_add_(0, self.pos, one)
            self.surface = torch.nonzero(links < 6)[:, 0]
            self.linked = torch.sort(self.neg * first + self.pos)[0]
            self.n = first
            self.pairs = None

    def temperature(self, t):
        T = self.amp * torch.sin(2 * float(np.float32(3.1415926)) * (t / self.period + self.phase))
        return torch.minimum(T, torch.zeros_like(T))

    def rest(self):
        v, l = self.site.shape[0], self.neg.shape[0]
        z = torch.zeros(v, 3, dtype=torch.float64, device=_DEV)
        q = torch.zeros(v, 4, dtype=torch.float64, device=_DEV)
        q[:, 0] = 1
        zl = torch.zeros(l, 3, dtype=torch.float64, device=_DEV)
        return [z, q, z.clone(), z.clone(), zl, zl.clone(), zl.clone()], (
            torch.ones(l, dtype=torch.bool, device=_DEV), torch.zeros(l, dtype=torch.bool, device=_DEV),
            torch.ones(v, dtype=torch.bool, device=_DEV))

    def ax(self, v):
        return torch.gather(v, 1, self.perm) * self.sx

    def unax(self, v):
        return torch.gather(v, 1, self.perm) * self.sb

    def links(self, u, q, P0, A0, B0, T, small, valid):
        L, n, p = self.L, self.neg, self.pos
        E = 2 * self.E[n] * self.E[p] / (self.E[n] + self.E[p])
        a2, b1, b2, b3 = E * L ** 3 / 12, E * L, E * L * L / 2, E * L ** 3 / 6
        quat = lambda x: torch.cat([x[:, :1], self.ax(x[:, 1:])], 1)  # noqa: E731
        R = _conj(quat(q[n]))
        B = _qmul(R, quat(q[p]))
        e = torch.zeros_like(P0)
        e[:, 0] = L
        at = _rot(R, self.ax(u[p] - u[n]) + e)
        rest = L / 2 * (2 + self.alpha * (T[n] + T[p]))
        ext = at[:, 0] - rest
        turn, extend = ((at[:, 1].abs() + at[:, 2].abs()) / at[:, 0]).detach(), (ext / rest).abs().detach()
        was = small
        small = torch.where(was, ~((turn > 1.2 * 0.05) | (extend > 1.2 * 0.5)), (turn < 0.05) & (extend < 0.5))
        valid = valid & (small == was)
        s = small[:, None]
        G = _to_x(at)
        one = torch.zeros_like(G)
        one[:, 0] = 1
        G = torch.where(s, one, G)
        B = torch.where(s, B, _qmul(G, B))
        zero = torch.zeros_like(ext)
        P = torch.where(s, torch.stack([ext, at[:, 1], at[:, 2]], 1),
                        torch.stack([at.norm(dim=1) - rest, zero, zero], 1))
        A1, A2 = _rotvec(G), _rotvec(B)

        def beam(axial, Px, P, X, Y, k, m2, m3):
            fx = axial * Px
            f = torch.stack([fx, k * P[:, 1] - m2 * (X[:, 2] + Y[:, 2]), k * P[:, 2] + m2 * (X[:, 1] + Y[:, 1])], 1)
            my = lambda i: torch.stack([torch.zeros_like(fx), -m2 * P[:, 2] - m3 * i(1), m2 * P[:, 1] - m3 * i(2)], 1)  # noqa: E731
            return f, my(lambda c: 2 * X[:, c] + Y[:, c]), my(lambda c: X[:, c] + 2 * Y[:, c])

        fN, mN, mP = beam(E * L * L / rest, P[:, 0], P, A1, A2, b1, b2, b3)
        tw = a2 * (A2[:, 0] - A1[:, 0])
        x = torch.zeros_like(fN)
        x[:, 0] = 1
        mN, mP = mN + tw[:, None] * x, mP - tw[:, None] * x
        fP = -fN
        dP, dA, dB = (P - P0) / 2, (A1 - A0) / 2, (A2 - B0) / 2
        dm = (2 * math.sqrt(self.mass) * self.zi) / self.dtl
        c, tN, tP = beam((E * L).sqrt(), dP[:, 0], dP, dA, dB, b1.sqrt(), (b2 * L / 2).sqrt(), (b3 * L * L / 6).sqrt())
        tw = (a2 * L * L / 6).sqrt() * (dB[:, 0] - dA[:, 0])
        v = valid[:, None].to(fN.dtype)
        fN, fP = fN + v * c * dm, fP - v * c * dm
        mN = mN + v * (tN + tw[:, None] * x) * (dm / 2)
        mP = mP + v * (tP - tw[:, None] * x) * (dm / 2)
        F, M = torch.zeros_like(u), torch.zeros_like(u)
        F = F.index_add(0, n, self.unax(_rot(_conj(G), fN))).index_add(0, p, self.unax(_rot(_conj(B), fP)))
        M = M.index_add(0, n, self.unax(_rot(_conj(G), mN))).index_add(0, p, self.unax(_rot(_conj(B), mP)))
        return F, M, P, A1, A2, small, torch.ones_like(valid)

    def contacts(self, u, p, T):
        """Contact forces between surface voxels that are not linked."""
        L, skin = self.L, 0.4 * self.L
        where = self.site * L + u
        if self.pairs is None or float((where - self.at).norm(dim=1).max()) > 0.49 * skin:
            self.at, self.pairs = where.clone(), self.list(where[self.surface], 1.25 * L + skin)
        i, j = self.pairs
        d = where[j] - where[i]
        far = d.norm(dim=1)
        size = L * (1 + self.alpha * T)
        depth = (size[i] + size[j]) * 0.625 - far
        hit = depth > 0
        i, j, d, far, depth = i[hit], j[hit], d[hit], far[hit], depth[hit]
        unit = d / far[:, None]
        ki, kj = 2 * self.E[i] * L, 2 * self.E[j] * L
        ci, cj = (self.zc * 2 * (self.mass * self.E[x] * L).sqrt() for x in (i, j))
        closing = ((p[i] - p[j]) / self.mass * unit).sum(1)
        f = unit * (2 / (1 / ki + 1 / kj) * depth + (ci + cj) / 2 * closing)[:, None]
        return torch.zeros_like(u).index_add(0, i, f).index_add(0, j, -f)

    def list(self, at, radius):
        """Pairs (lower, higher voxel) of surface voxels of one robot within radius, not linked."""
        cell = torch.floor(at / radius).to(torch.int64)
        cell = cell - cell.amin(0) + 1
        span = cell.amax(0) + 2
        rob = self.rob[self.surface]
        key = lambda c: ((rob * span[0] + c[:, 0]) * span[1] + c[:, 1]) * span[2] + c[:, 2]  # noqa: E731
        order = torch.argsort(key(cell))
        keys = key(cell)[order]
        found = []
        for dx in (-1, 0, 1):
            for dy in (-1, 0, 1):
                for dz in (-1, 0, 1):
                    near = key(cell + torch.tensor([dx, dy, dz], device=_DEV))
                    a, b = torch.searchsorted(keys, near), torch.searchsorted(keys, near, right=True)
                    count = b - a
                    me = torch.repeat_interleave(torch.arange(len(near), device=_DEV), count)
                    k = torch.arange(len(me), device=_DEV) - torch.repeat_interleave(count.cumsum(0) - count, count) + a[me]
                    other = order[k]
                    keep = (me < other) & ((at[me] - at[other]).norm(dim=1) < radius)
                    found.append(torch.stack([self.surface[me[keep]], self.surface[other[keep]]]))
        i, j = torch.cat(found, 1)
        k = i * self.n + j
        pos = torch.searchsorted(self.linked, k).clamp(max=max(0, len(self.linked) - 1))
        free = self.linked[pos] != k if len(self.linked) else torch.ones_like(k, dtype=torch.bool)
        return i[free], j[free]

    def step(self, state, flags, T, TT=None):
        u, q, p, h, P, A, B = state
        small, valid, stick = flags
        F, M, P, A, B, small, valid = self.links(u, q, P, A, B, T, small, valid)
        f = _rot(q, F)
        vel = p / self.mass
        f = f - vel * (self.zg * 2 * (self.mass * self.E * self.L).sqrt())[:, None]
        f = f + torch.tensor([0.0, 0.0, self.grav], dtype=torch.float64, device=_DEV)
        c_floor = self.zc * 2 * (self.mass * self.E * self.L).sqrt()
        pen = self.L * T * self.alpha / 2 - self.site[:, 2] * self.L - u[:, 2]
        if self.diff:
            x = pen / 1e-4
            N = 1e5 * 1e-4 * torch.nn.functional.softplus(x, threshold=1e9)
            slow = (vel[:, 0] ** 2 + vel[:, 1] ** 2 + 1e-6).sqrt()
            g = (self.mu_k * N / slow)[:, None]
            f = f + torch.cat([-g * vel[:, :2], (N - c_floor * vel[:, 2] * torch.sigmoid(x))[:, None]], 1)
            p = p + f * self.dt
            move = p * (self.dt / self.mass)
        else:
            if self.collide:
                f = f - self.contacts(u, p, T)
            floor = pen >= 0
            N = 2 * self.E * self.L * pen
            cur = f + torch.cat([torch.zeros_like(f[:, :2]), (floor * (N - c_floor * vel[:, 2]))[:, None]], 1)
            slip = (cur[:, 0] ** 2 + cur[:, 1] ** 2) > (self.mu_s * N) ** 2
            was = stick
            stick = floor & stick & ~slip
            flat = torch.cat([vel[:, :2], torch.zeros_like(vel[:, :1])], 1)
            fast = flat.norm(dim=1, keepdim=True)
            drag = flat / torch.where(fast > 0, fast, torch.ones_like(fast)) * (self.mu_k * N)[:, None]
            cur = cur - drag * (floor & ~was)[:, None]
            p = p + cur * self.dt
            move = p * (self.dt / self.mass)
            left = ((cur - f)[:, :2] * move[:, :2]).sum(1) + 0.5 / self.mass * (p[:, :2] ** 2).sum(1)
            stick = torch.where(floor, stick | (left <= 0), stick)
            held = (floor & stick)[:, None] & torch.tensor([True, True, False], device=_DEV)
            p, move = torch.where(held, 0.0, p), torch.where(held, 0.0, move)
        u = u + move
        m = _rot(q, M) - h / self.inertia * (self.zg * 2 * (self.inertia * self.E * self.L ** 3).sqrt())[:, None]
        h = h + m * self.dt
        q = _qmul(_from_rotvec(h * (self.dt / self.inertia)), q)
        q = q / q.norm(dim=1, keepdim=True)
        if not self.diff:
            after = self.L * T * self.alpha / 2 - self.site[:, 2] * self.L - u[:, 2] >= 0
            h = torch.where((after & stick)[:, None], 0.0, h)
        return [u, q, p, h, P, A, B], (small, valid, stick)


def exact(case, seed):
    if case.get("extras"):
        return None
    problems = _problems(case, seed)
    if case["kind"] != "diff":
        body = _Body(problems)
        with torch.no_grad():
            state, flags = body.rest()
            t = torch.zeros_like(body.phase)
            for _ in range(case["steps"]):
                state, flags = body.step(state, flags, body.temperature(t))
                t = t + body.dt[:, 0]
        u, q, p, h = state[:4]
        at = (body.site * body.L + u).cpu().numpy()
        if case["kind"] == "run":
            n = np.bincount(body.rob.cpu().numpy())
            mean = lambda a: np.stack([np.bincount(body.rob.cpu().numpy(), a[:, k]) / n for k in range(3)], 1)  # noqa: E731
            com = mean(at)
            return dict(pos=at, fitness=com[:, 0] - mean(body.site.cpu().numpy() * body.L)[:, 0], com=com, steps=None, history=None)
        return dict(pos=at, quat=q.cpu().numpy(), linmom=p.cpu().numpy(), angmom=h.cpu().numpy())
    kind = torch.float32 if case["bits"] == 32 else torch.float64
    phase = np.concatenate([p["phase"] for p in problems])
    logE = np.log10(np.concatenate([p["voxel_E"] for p in problems]).astype(np.float64))
    psi = torch.tensor(phase * 2 * math.pi, dtype=kind).double().to(_DEV).requires_grad_(True)
    logE = torch.tensor(logE, dtype=kind).double().to(_DEV).requires_grad_(True)
    base = _Body(problems, diff=True)
    kept = []

    def one(state, flags, n):
        body = base
        body.phase, body.E = psi / (2 * math.pi), 10.0 ** logE
        return body.step(state, flags, body.temperature(times[n]))

    dt = float(base.dt[0, 0])
    times = [0.0]
    for _ in range(case["steps"]):
        times.append(times[-1] + dt)
    state, flags = base.rest()
    with torch.no_grad():
        for n in range(case["steps"]):
            kept.append((state, flags))
            state, flags = one(state, flags, n)
    weight = torch.tensor(np.concatenate([np.full(len(p["phase"]), -1.0 / len(p["phase"])) for p in problems]), device=_DEV)
    bar = [torch.zeros_like(x) for x in state]
    bar[0][:, 0] = weight
    at = (base.site * base.L + state[0]).detach().cpu()
    gpsi, gE = torch.zeros_like(psi), torch.zeros_like(logE)
    for n in reversed(range(case["steps"])):
        into = [x.detach().requires_grad_(True) for x in kept[n][0]]
        got, _ = one(into, kept[n][1], n)
        grads = torch.autograd.grad(got, into + [psi, logE], grad_outputs=bar, allow_unused=True)
        bar = [torch.zeros_like(x) if g is None else g for x, g in zip(into, grads)]
        gpsi, gE = gpsi + grads[-2], gE + grads[-1]
        kept.pop()
    return dict(pos=at, psi=gpsi.detach().cpu(), logE=gE.detach().cpu())
