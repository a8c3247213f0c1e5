"""The work that users of this framework have it do, as timed cases.

Every case goes through the public Python API (voxelyze_amd.api, voxelyze_amd.adjoint) as a
program written against it does: a model is built in bulk, run for a moment (so that it is on the
device, with its launch shapes settled) and saved as a checkpoint; one pass restores that
checkpoint, steps, and reads the result.

kind        what it stands for
beam        a small body under load: a viewer or controller that steps and reads every frame
            (calls > 1, no restore), or one rollout; optionally with a Poisson's ratio
lattice     one large body of two materials, falling or lying on the floor with friction
robots      a population of actuated robots, each with its own shape and phases, evaluated in one
            batch (positions and centres of mass are what an optimiser scores)
porous      a plastic porous block crushed by a prescribed displacement, with self-collision
gradient    one training step: rollout, loss on the centres of mass, gradients with respect to
            every voxel's modulus and actuation phase
static      the static linear solve of a loaded block

exact() restates the same model in plain torch in 64 bits.
"""
import math

import numpy as np
import torch

from voxelyze_amd import adjoint, workloads
from voxelyze_amd.api import CVoxelyze, MIXED

PITCH = 0.005
WARM = 26          # steps before the saved state: the launch shapes settle in the first 24
FUSED_FP64 = 2     # setPrecision: the FP64 reference of the mixed step and its adjoint
PRECISION = {"fp64": 0, "mixed": MIXED, "fused64": FUSED_FP64}


def listed():
    return [
        # a GUI or control loop around a small cantilever: step once, read every position
        {"name": "beam_frames", "kind": "beam", "nx": 20, "ny": 4, "nz": 4, "nu": 0.0, "precision": "fp64",
         "calls": 32, "steps": 1},
        # the 320-voxel cantilever rolled out in one call
        {"name": "beam_rollout", "kind": "beam", "nx": 20, "ny": 4, "nz": 4, "nu": 0.0, "precision": "fp64",
         "calls": 1, "steps": 1000},
        # a ragged bar in mixed precision
        {"name": "bar_mixed", "kind": "beam", "nx": 37, "ny": 11, "nz": 7, "nu": 0.0, "precision": "mixed",
         "calls": 1, "steps": 1000},
        # nearly incompressible rubber: the volumetric terms of a Poisson's ratio
        {"name": "bar_poisson", "kind": "beam", "nx": 43, "ny": 15, "nz": 13, "nu": 0.35, "precision": "fp64",
         "calls": 1, "steps": 400},
        # a mid-size body lying on the floor, odd sizes
        {"name": "lattice_mid", "kind": "lattice", "nx": 47, "ny": 37, "nz": 29, "lift": 0, "precision": "fp64",
         "steps": 400},
        # the largest single body: the 128 x 128 x 64-site drop lattice
        {"name": "lattice_fp64", "kind": "lattice", "nx": 128, "ny": 128, "nz": 64, "lift": 2, "precision": "fp64",
         "steps": 300},
        {"name": "lattice_mixed", "kind": "lattice", "nx": 101, "ny": 97, "nz": 53, "lift": 2, "precision": "mixed",
         "steps": 400},
        # populations: thousands of small bodies in mixed precision; fewer, checked in FP64
        {"name": "robots_mixed", "kind": "robots", "robots": 160, "vmin": 100, "vmax": 8000, "precision": "mixed",
         "steps": 200},
        {"name": "robots_fp64", "kind": "robots", "robots": 48, "vmin": 100, "vmax": 3000, "precision": "fp64",
         "steps": 200},
        # self-collision and plasticity
        {"name": "porous_fp64", "kind": "porous", "n": 40, "precision": "fp64", "steps": 150},
        # gradients of a rollout, 32 x 32 x 16-site bodies
        {"name": "gradient_mixed", "kind": "gradient", "robots": 8, "nx": 32, "ny": 32, "nz": 16,
         "precision": "mixed", "steps": 200, "every": 50},
        # static equilibrium of a loaded block
        {"name": "static_block", "kind": "static", "nx": 60, "ny": 44, "nz": 30},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["beam", "beam", "lattice", "lattice", "robots", "robots", "porous", "gradient", "static"])
    both = rng.choice(["fp64", "mixed"])
    if kind == "beam":
        nu = rng.choice([0.0, 0.0, round(rng.uniform(0.1, 0.4), 2)])
        calls = rng.choice([1, 1, _log_int(rng, 8, 64)])
        return {"kind": kind, "nx": _log_int(rng, 6, 50), "ny": _log_int(rng, 2, 16), "nz": _log_int(rng, 2, 14),
                "nu": nu, "precision": "fp64" if nu else both, "calls": calls,
                "steps": _log_int(rng, 1, 10) if calls > 1 else _log_int(rng, 100, 1000)}
    if kind == "lattice":
        return {"kind": kind, "nx": _log_int(rng, 15, 110), "ny": _log_int(rng, 15, 110), "nz": _log_int(rng, 9, 60),
                "lift": rng.choice([0, 2]), "precision": both, "steps": _log_int(rng, 100, 400)}
    if kind == "robots":
        vmin = _log_int(rng, 50, 400)
        return {"kind": kind, "robots": _log_int(rng, 4, 160), "vmin": vmin, "vmax": vmin + _log_int(rng, 50, 7000),
                "precision": both, "steps": _log_int(rng, 50, 200)}
    if kind == "porous":
        return {"kind": kind, "n": _log_int(rng, 16, 48), "precision": both, "steps": _log_int(rng, 50, 150)}
    if kind == "gradient":
        return {"kind": kind, "robots": _log_int(rng, 1, 8), "nx": rng.randint(8, 32), "ny": rng.randint(8, 32),
                "nz": rng.randint(6, 16), "precision": rng.choice(["mixed", "mixed", "fused64"]),
                "steps": _log_int(rng, 40, 200), "every": rng.choice([20, 25, 50])}
    return {"kind": kind, "nx": _log_int(rng, 8, 64), "ny": _log_int(rng, 6, 48), "nz": _log_int(rng, 4, 32)}


# ------------------------------------------------------------------------------- the models
# A model is plain data, made from the case and the seed alone: `mats` (material properties),
# `robots` (per robot: lattice sites and material indices, in the order the voxels are added),
# the supports and loads, the environment and the time step.  How many voxels there are is the
# case's; which sites, materials, phases, moduli and loads are the seed's.

def _box(nx, ny, nz):
    s = np.arange(nx * ny * nz)
    return np.stack([s % nx, (s // nx) % ny, s // (nx * ny)], 1).astype(np.int32)


def _sorted(ijk):
    """lattice order: x fastest"""
    return ijk[np.lexsort((ijk[:, 0], ijk[:, 1], ijk[:, 2]))].astype(np.int32)


def _robot_sizes(case):
    """sizes spread evenly over [vmin, vmax], in a fixed shuffled order"""
    R, lo, hi = case["robots"], case["vmin"], case["vmax"]
    sizes = [lo + int((r + 0.5) / R * (hi - lo)) for r in range(R)]
    return [sizes[i] for i in np.random.default_rng(R).permutation(R)]


def _time_step(mats, fraction):
    """A fraction of the oscillation limit of the stiffest, lightest link; a float, as the API takes it."""
    w2 = max(m["E"] / m["rho"] for m in mats) / PITCH ** 2
    return float(np.float32(fraction / (2 * math.pi * math.sqrt(w2))))


def _model(case, seed):
    rng = np.random.default_rng([seed, 77])
    kind = case["kind"]
    M = {"gravity": 0.0, "floor": False, "contacts": False, "fixed": np.zeros(0, int), "loads": None,
         "ramp": None, "phase": None, "act": None, "fraction": 0.9}
    if kind in ("beam", "static"):
        nx, ny, nz = case["nx"], case["ny"], case["nz"]
        ijk = _box(nx, ny, nz)
        M["mats"] = [{"E": 1e6, "rho": 1000.0, "nu": case.get("nu", 0.0)}]
        M["robots"] = [(ijk, np.zeros(len(ijk), np.int32))]
        ax, end = (0, nx - 1) if kind == "beam" else (2, nz - 1)
        M["fixed"] = np.nonzero(ijk[:, ax] == 0)[0]
        tips = np.nonzero(ijk[:, ax] == end)[0]
        # a load on the free end whose size, direction and distribution differ by seed
        each = rng.normal(size=3) * (5e-4 if kind == "beam" else 2e-5) * 1e6 * PITCH ** 2
        M["loads"] = (tips, (each[None, :] * (rng.random(len(tips)) + 0.5)[:, None]).astype(np.float32))
        if M["mats"][0]["nu"]:
            M["fraction"] = 0.4
    elif kind == "lattice":
        ijk = _box(case["nx"], case["ny"], case["nz"])
        n = len(ijk)
        occ = np.sort(rng.permutation(n)[:int(0.9 * n)])
        ijk = ijk[occ]
        ijk[:, 2] += case["lift"]
        mat = (rng.random(len(occ)) < 0.3).astype(np.int32)
        fr = {"mus": 1.0, "muk": 0.5}
        M["mats"] = [{"E": 1e6, "rho": 1000.0, **fr}, {"E": 1e7, "rho": 1500.0, **fr}]
        M["robots"] = [(ijk, mat)]
        M["gravity"], M["floor"] = 1.0, True
    elif kind in ("robots", "gradient"):
        fr = {"mus": 1.0, "muk": 0.5, "rho": 1000.0}
        if kind == "robots":
            M["mats"] = [{"E": 1e5, **fr}, {"E": 1e7, **fr}, {"E": 1e6, "cte": 0.01, **fr}, {"E": 1e6, "cte": -0.01, **fr}]
            shapes = [workloads.grow_robot_native(1000 * int(seed) + r, n) for r, n in enumerate(_robot_sizes(case))]
            for g in shapes:
                g[:, 2] -= g[:, 2].min()
            M["robots"] = [(_sorted(g), rng.integers(0, 4, len(g)).astype(np.int32)) for g in shapes]
        else:
            M["mats"] = [{"E": 1e6, **fr}, {"E": 1e6, "cte": 0.01, **fr}, {"E": 1e6, "cte": -0.01, **fr}]
            shapes = [workloads.random_fill_robot(5, r, case["nx"], case["ny"], case["nz"])[0] for r in range(case["robots"])]
            M["robots"] = [(g, rng.integers(0, 3, len(g)).astype(np.int32)) for g in shapes]
        total = sum(len(i) for i, _ in M["robots"])
        M["phase"] = rng.uniform(0, 2 * math.pi, total).astype(np.float32)
        M["act"] = (39.0, 2.0)
        M["gravity"], M["floor"] = 1.0, True
        if kind == "gradient":
            M["modulus"] = (1e6 * np.exp(rng.uniform(-0.2, 0.2, total))).astype(np.float32)
            M["fraction"] = 0.7
    elif kind == "porous":
        n = case["n"]
        solid = np.ones((n, n, n), dtype=bool)   # [z, y, x]
        g, void = np.arange(n), np.random.default_rng(3)
        while 1.0 - solid.mean() < 0.2:
            c, r = void.random(3) * n, void.integers(2, 7)
            solid &= ((g[:, None, None] - c[0]) ** 2 + (g[None, :, None] - c[1]) ** 2 + (g[None, None, :] - c[2]) ** 2) > r * r
        solid = workloads.largest_component(solid)
        for a in (1, 2):   # the block as it is or mirrored
            if rng.random() < 0.5:
                solid = np.flip(solid, a)
        z, y, x = np.nonzero(solid)
        ijk = np.stack([x, y, z], 1).astype(np.int32)
        M["mats"] = [{"E": 5e6, "rho": 1000.0, "plastic": (5e5, 2.5e5, 3.75e5)}]
        M["robots"] = [(ijk, np.zeros(len(ijk), np.int32))]
        M["fixed"] = np.nonzero(ijk[:, 2] == 0)[0]
        top = np.nonzero(ijk[:, 2] == n - 1)[0]
        M["contacts"] = True
        M["ramp"] = (top, rng.uniform(4e-3, 6e-3) * PITCH)   # 0.4 to 0.6 % of a pitch a step, downwards
    M["dt"] = _time_step(M["mats"], M["fraction"])
    return M


def _build(case, M):
    sim = CVoxelyze(PITCH)
    mats = []
    for p in M["mats"]:
        m = sim.addMaterial(p["E"], p["rho"])
        if "plastic" in p:
            m.setModelBilinear(p["E"], *p["plastic"])
        m.setPoissonsRatio(p.get("nu", 0.0))
        m.setCte(p.get("cte", 0.0))
        m.setStaticFriction(p.get("mus", 0.0))
        m.setKineticFriction(p.get("muk", 0.0))
        mats.append(m.index)
    sim.setGravity(M["gravity"])
    sim.enableFloor(M["floor"])
    for r, (ijk, mat) in enumerate(M["robots"]):
        if r:
            sim.addRobot()
        sim.setVoxels(np.asarray(mats, np.int32)[mat], ijk)
    for i in M["fixed"]:
        sim.voxel(int(i)).external().setFixedAll()
    if M["loads"]:
        for i, f in zip(*M["loads"]):
            sim.voxel(int(i)).external().setForce(float(f[0]), float(f[1]), float(f[2]))
    if M["ramp"]:
        top, per_step = M["ramp"]
        for i in top:
            sim.voxel(int(i)).external().setDisplacementRamp((0, 0, 0), (0, 0, -per_step / M["dt"]))
    if M["contacts"]:
        sim.enableCollisions(True)
    if M["act"]:
        sim.setActuation(True, 0.0, *M["act"])
        sim.setPhases(M["phase"])
    sim.setPrecision(PRECISION[case.get("precision", "fp64")])
    return sim


def prepare(case, seed):
    M = _model(case, seed)
    sim = _build(case, M)
    s = {"sim": sim, "case": case, "dt": M["dt"]}
    if case["kind"] == "static":
        sim.robotCom()   # the model is on the device
        return s
    if case["kind"] == "gradient":
        s["log_modulus"] = torch.from_numpy(np.log(M["modulus"].astype(np.float64))).cuda().requires_grad_()
        s["phase"] = torch.from_numpy(M["phase"].astype(np.float64)).cuda().requires_grad_()
    s["dts"] = np.full(sim.robotCount(), M["dt"], np.float32)
    sim.robotStep(WARM, s["dts"])
    sim.checkpointSave(0)
    return s


def run(s):
    sim, case, dt = s["sim"], s["case"], s["dt"]
    kind = case["kind"]
    if kind == "static":
        if not sim.doLinearSolve():
            raise RuntimeError(sim.lastError())
        st = sim.state()
        return {"pos": st["pos"], "orient": st["orient"]}
    if kind == "gradient":
        pos = adjoint.rollout(sim, s["log_modulus"], s["phase"], case["steps"], every=case["every"], dt=dt)
        loss = -adjoint.robot_com(sim, pos)[:, 0].sum()
        s["log_modulus"].grad = s["phase"].grad = None
        loss.backward()
        return {"pos": pos.detach(), "d_log_modulus": s["log_modulus"].grad, "d_phase": s["phase"].grad}
    if kind == "beam" and case["calls"] > 1:
        for _ in range(case["calls"]):
            if case["steps"] == 1:
                sim.doTimeStep(dt)
            else:
                sim.step(dt, case["steps"])
            pos = sim.positions()
        return {"pos": pos}
    sim.checkpointRestore(0)
    if kind == "robots":
        sim.robotStep(case["steps"], s["dts"])
        return {"com": sim.robotCom(), "pos": sim.positions()}
    sim.step(dt, case["steps"])
    if case["precision"] == "fp64" and kind in ("beam", "porous"):
        return sim.state()   # everything, flags among it: small enough to read whole
    return {"pos": sim.positions()}


# ------------------------------------------------------------------------------------- work
# Bytes: what a step reads and writes where a body's state does not stay on the chip (FP64: 300
# per voxel and 384 per link; mixed 300 and 212), once a pass where it does (256 MB of cache);
# operations: about 450 per link and 250 per voxel and step, three times that and a recompute
# for a gradient.

ON_CHIP = 256e6


def _counts(case):
    k = case["kind"]
    if k in ("beam", "static"):
        nx, ny, nz = case["nx"], case["ny"], case["nz"]
        return nx * ny * nz, 3 * nx * ny * nz - nx * ny - ny * nz - nz * nx
    if k == "lattice":
        n = 0.9 * case["nx"] * case["ny"] * case["nz"]
        return n, 2.67 * n
    if k == "robots":
        n = case["robots"] * 0.5 * (case["vmin"] + case["vmax"])
        return n, 2.65 * n
    if k == "porous":
        n = 0.79 * case["n"] ** 3
        return n, 2.6 * n
    n = 0.7 * case["robots"] * case["nx"] * case["ny"] * case["nz"]
    return n, 2.0 * n


def work(case):
    v, l = _counts(case)
    if case["kind"] == "static":
        it = 9 * max(case["nx"], case["ny"], case["nz"])   # iterations of a conjugate gradient
        return {"bytes": 220.0 * v, "flops": it * (72.0 * l + 100.0 * v)}
    steps = case["steps"] * case.get("calls", 1)
    step = 300 * v + (212 if case["precision"] == "mixed" else 384) * l
    flops = steps * (450 * l + 250 * v)
    if case["kind"] == "gradient":
        return {"bytes": 3.0 * steps * step, "flops": 5.0 * flops}
    return {"bytes": float(step * (steps if step > ON_CHIP else 1) + 24 * v * case.get("calls", 1)),
            "flops": float(flops)}


# ------------------------------------------------------------------- the same in 64 bits, plainly

def _dev():
    return "cuda" if torch.cuda.is_available() else "cpu"


def _t(x, dtype=torch.float64):
    return torch.as_tensor(np.ascontiguousarray(x)).to(_dev(), dtype)


def _qmul(a, b):
    aw, av, bw, bv = a[:, :1], a[:, 1:], b[:, :1], b[:, 1:]
    return torch.cat([aw * bw - (av * bv).sum(1, True), aw * bv + bw * av + torch.linalg.cross(av, bv)], 1)


def _conj(q):
    return torch.cat([q[:, :1], -q[:, 1:]], 1)


def _rot(q, v):
    """q v q* (not assuming a unit quaternion)"""
    w, u = q[:, :1], q[:, 1:]
    return (w * w - (u * u).sum(1, True)) * v + 2 * (u * v).sum(1, True) * u + 2 * w * torch.linalg.cross(u, v)


def _to_vector(q):
    """quaternion to rotation vector; (2 - 2 w)/(1 - w^2) is 2/(1 + w)"""
    w = q[:, :1]
    s = 1 - w * w
    near = 2 * torch.sqrt(2 / (1 + w))
    if not bool((s >= 2.4e-3).any()):
        return q[:, 1:] * near
    sf = torch.where(s < 2.4e-3, torch.ones_like(s), s)
    far = 2 * torch.acos(torch.where(s < 2.4e-3, torch.zeros_like(w), w)) / torch.sqrt(sf)
    return q[:, 1:] * torch.where(s < 2.4e-3, near, far)


def _from_vector(v):
    h = 0.5 * v
    m2 = (h * h).sum(1, True)
    tiny = m2 * m2 < 5.328e-15
    m = torch.sqrt(torch.where(tiny, torch.ones_like(m2), m2))
    w = torch.where(tiny, 1 - 0.5 * m2, torch.cos(m))
    return torch.cat([w, h * torch.where(tiny, 1 - m2 / 6, torch.sin(m) / m)], 1)


def _angle_to_x(d):
    """the rotation that takes d onto the x axis"""
    yx, zx = d[:, 1:2] / d[:, :1], d[:, 2:] / d[:, :1]
    near = (yx.abs() < 1.732e-2) & (zx.abs() < 1.732e-2)
    z = torch.zeros_like(yx)
    qn = torch.cat([1 - 0.125 * (yx * yx + zx * zx), z, 0.5 * zx, -0.5 * yx], 1)
    ds = torch.where(near, torch.tensor([1.0, 1.0, 0.0], dtype=d.dtype, device=d.device), d)
    n = ds / ds.norm(dim=1, keepdim=True)
    half = 0.5 * torch.acos(n[:, :1].clamp(-1, 1))
    a = torch.sin(half) / torch.sqrt(n[:, 1:2] ** 2 + n[:, 2:] ** 2)
    return torch.where(near, qn, torch.cat([torch.cos(half), z, n[:, 2:] * a, -n[:, 1:2] * a], 1))


class _Exact:
    """The explicit step on plain arrays."""

    def __init__(self, M):
        self.M, mats = M, M["mats"]
        ijk = np.concatenate([i for i, _ in M["robots"]]).astype(np.int64)
        rob = np.repeat(np.arange(len(M["robots"])), [len(i) for i, _ in M["robots"]])
        self.ijk = ijk
        self.n = n = len(ijk)
        mat = np.concatenate([m for _, m in M["robots"]]).astype(np.int64)
        lo, hi = ijk.min(0) - 1, ijk.max(0) + 2
        dim = hi - lo

        def key(p):
            p = p - lo
            return ((rob * dim[2] + p[:, 2]) * dim[1] + p[:, 1]) * dim[0] + p[:, 0]
        k = key(ijk)
        order = np.argsort(k)
        ks = k[order]
        neg, pos, self.span = [], [], []
        inside = np.ones(n, bool)
        for a in range(3):
            for sign in (1, -1):
                step = np.zeros(3, np.int64)
                step[a] = sign
                q = key(ijk + step)
                at = np.minimum(np.searchsorted(ks, q), n - 1)
                has = ks[at] == q
                inside &= has
                if sign == 1:
                    i = np.nonzero(has)[0]
                    self.span.append((sum(map(len, neg)), sum(map(len, neg)) + len(i)))
                    neg.append(i)
                    pos.append(order[at[has]])
        self.neg, self.pos_ = np.concatenate(neg), np.concatenate(pos)
        self.N, self.P = _t(self.neg, torch.long), _t(self.pos_, torch.long)
        self.surface = ~inside

        def per(name, default=0.0):
            return _t(np.array([float(np.float32(m.get(name, default))) for m in mats])[mat])[:, None]
        self.L = L = PITCH
        self.rho, self.nu, self.cte = per("rho"), per("nu"), per("cte")
        self.mus, self.muk = per("mus"), per("muk")
        self.E0 = per("E")
        self.plastic = mats[0].get("plastic")
        self.mass = self.rho * L ** 3
        self.inertia = self.mass * L * L / 6
        self.fixed = _t(M["fixed"], torch.long)
        self.free = torch.ones(n, 1, dtype=torch.bool, device=_dev())
        if len(M["fixed"]):
            self.free[self.fixed] = False
        self.ext = torch.zeros(n, 3, dtype=torch.float64, device=_dev())
        if M["loads"]:
            self.ext[_t(M["loads"][0], torch.long)] = _t(M["loads"][1])
        self.x0 = _t(ijk) * L
        self.ramp = _t(M["ramp"][0], torch.long) if M["ramp"] else None
        if self.ramp is not None:
            self.free[self.ramp] = False
        if M["contacts"]:
            self._pairs()

    def _pairs(self):
        """pairs of surface voxels that can touch: within 2.5 pitches at rest and not joined by a
        path of five links or fewer"""
        ijk = self.ijk
        R = 5
        dim = ijk.max(0) + 1 + 2 * R
        solid = np.full(dim, -1, np.int64)
        solid[tuple((ijk + R).T)] = np.arange(self.n)
        solid = _t(solid, torch.long)
        c = _t(ijk + R, torch.long)

        def there(o):
            return solid[c[:, 0] + o[0], c[:, 1] + o[1], c[:, 2] + o[2]]
        full = {(0, 0, 0): torch.ones(self.n, dtype=torch.bool, device=_dev())}
        at = {}
        reach = dict(full)
        for _ in range(5):
            nxt = {o: r.clone() for o, r in reach.items()}
            for o, r in reach.items():
                for a in range(3):
                    for s in (1, -1):
                        p = tuple(o[b] + (s if a == b else 0) for b in range(3))
                        if p not in at:
                            at[p] = there(p) >= 0
                        new = r & at[p]
                        nxt[p] = nxt[p] | new if p in nxt else new
            reach = nxt
        surf = _t(self.surface, torch.bool)
        I, J = [], []
        for x in range(-2, 3):
            for y in range(-2, 3):
                for z in range(-2, 3):
                    if (x, y, z) <= (0, 0, 0) or x * x + y * y + z * z > 6.25:
                        continue
                    j = there((x, y, z))
                    ok = (j >= 0) & surf & surf[j.clamp(min=0)]
                    if (x, y, z) in reach:
                        ok &= ~reach[(x, y, z)]
                    I.append(torch.nonzero(ok)[:, 0])
                    J.append(j[I[-1]])
        self.ci, self.cj = torch.cat(I), torch.cat(J)

    def to_x(self, v):
        (a, b), (c, d), (e, f) = self.span
        y, z = v[c:d], v[e:f]
        return torch.cat([v[a:b], torch.stack([y[:, 1], -y[:, 0], y[:, 2]], 1), torch.stack([z[:, 2], z[:, 1], -z[:, 0]], 1)])

    def from_x(self, v):
        (a, b), (c, d), (e, f) = self.span
        y, z = v[c:d], v[e:f]
        return torch.cat([v[a:b], torch.stack([-y[:, 1], y[:, 0], y[:, 2]], 1), torch.stack([-z[:, 2], z[:, 1], z[:, 0]], 1)])

    def to_xq(self, q):
        return torch.cat([q[:, :1], self.to_x(q[:, 1:])], 1)

    def start(self):
        n, m = self.n, len(self.neg)
        z = lambda k, c, **o: torch.zeros(k, c, device=_dev(), **({"dtype": torch.float64} | o))  # noqa: E731
        q = z(n, 4)
        q[:, 0] = 1
        return {"pos": self.x0.clone(), "q": q, "lin": z(n, 3), "ang": z(n, 3), "static": ~z(n, 1, dtype=torch.bool),
                "p2": z(m, 3), "a1": z(m, 3), "a2": z(m, 3), "small": ~z(m, 1, dtype=torch.bool), "lvv": z(m, 1, dtype=torch.bool),
                "strain": z(m, 1), "top": z(m, 1), "off": z(m, 1), "t": 0.0}

    def constants(self, E=None):
        """link and voxel constants of the voxels' moduli"""
        L, E = self.L, self.E0 if E is None else E
        e1, e2 = E[self.N], E[self.P]
        k = {"E": 2 * e1 * e2 / (e1 + e2)}
        nu = torch.zeros_like(k["E"])
        k["hat"] = k["E"]
        if bool((self.nu != 0).any()):
            hat = E / ((1 - 2 * self.nu) * (1 + self.nu))
            k["hat"] = 2 * hat[self.N] * hat[self.P] / (hat[self.N] + hat[self.P])
            nu = torch.sqrt((k["hat"] - k["E"]) / (2 * k["hat"]) + 0.0625) - 0.25
            k["hat"] = k["E"] / ((1 - 2 * nu) * (1 + nu))
        k["nu"] = nu
        Ek = k["E"]
        k["a2"], k["b1"], k["b2"], k["b3"] = Ek * L ** 3 / (12 * (1 + nu)), Ek * L, Ek * L ** 2 / 2, Ek * L ** 3 / 6
        k["sA1"], k["sA2"] = torch.sqrt(Ek * L), torch.sqrt(k["a2"] * L * L / 6)
        k["sB2"], k["sB3"] = torch.sqrt(k["b2"] * L / 2), torch.sqrt(k["b3"] * L * L / 6)
        k["damp"] = 2 * torch.sqrt(self.mass)     # internal damping ratio 1
        k["pen"] = 2 * E * L
        return k

    def step(self, s, k, dt, prev, phase=None):
        M, L, N, P = self.M, self.L, self.N, self.P
        # temperatures, rest lengths
        f = torch.ones(self.n, 1, dtype=torch.float64, device=_dev())
        if M["act"]:
            amp, freq = M["act"]
            f = 1 + self.cte * (amp * torch.sin(2 * math.pi * freq * s["t"] + phase))
        rest = 0.5 * L * (f[N] + f[P])
        # links
        d = self.to_x(s["pos"][P] - s["pos"][N])
        a1, a2 = self.to_xq(s["q"][N]), self.to_xq(s["q"][P])
        tr = _conj(a1)
        d, a2 = _rot(tr, d), _qmul(tr, a2)
        turn, ext = (d[:, 1:2].abs() + d[:, 2:].abs()) / d[:, :1], (1 - d[:, :1] / rest).abs()
        small = s["small"]
        shrink, grow = ~small & (turn < 0.05) & (ext < 0.5), small & ((turn > 0.06) | (ext > 0.6))
        small = (small | shrink) & ~grow
        lvv = s["lvv"] & ~(shrink | grow)
        first = torch.zeros_like(a1)
        first[:, 0] = 1
        p2, r1, r2, e2 = torch.cat([d[:, :1] - rest, d[:, 1:]], 1), torch.zeros_like(d), _to_vector(a2), a2
        big = not bool(small.all())
        if big:
            ds = torch.where(small, torch.tensor([1.0, 0.1, 0.1], dtype=d.dtype, device=d.device), d)
            first = torch.where(small, first, _angle_to_x(ds))
            e2 = torch.where(small, a2, _qmul(first, a2))
            p2 = torch.where(small, p2, torch.cat([ds.norm(dim=1, keepdim=True) - rest, torch.zeros_like(d[:, 1:])], 1))
            r1, r2 = torch.where(small, r1, _to_vector(first)), _to_vector(e2)
        strain = p2[:, :1] / rest
        top, off = torch.maximum(s["top"], strain), s["off"]
        area = torch.full_like(strain, L * L)
        if self.plastic:
            E = self.E0[0]
            Ep, ys, fs = self.plastic
            ey = ys / E
            efail = (fs - (ys - Ep * ey)) / Ep
            curve = torch.where(strain <= ey, E * strain, ys + Ep * (strain - ey))
            curve = torch.where(strain > efail, torch.zeros_like(curve), curve)
            rising = strain > s["top"]
            off = torch.where(rising, top - curve / E, off)
            stress = torch.where(rising, curve, E * (strain - off))
            alive = top <= efail
        else:
            stress, alive = k["E"] * strain, None
            if bool((self.nu != 0).any()):
                tss, area = self.transverse(s)
                stress = k["hat"] * ((1 - k["nu"]) * strain + k["nu"] * tss)
        py, pz = p2[:, 1:2], p2[:, 2:]
        (y1, z1, x1), (y2, z2, x2) = [(r[:, 1:2], r[:, 2:], r[:, :1]) for r in (r1, r2)]
        a_, b1, b2, b3 = k["a2"], k["b1"], k["b2"], k["b3"]
        fN = torch.cat([stress * area, b1 * py - b2 * (z1 + z2), b1 * pz + b2 * (y1 + y2)], 1)
        fP = -fN
        mN = torch.cat([a_ * (x2 - x1), -b2 * pz - b3 * (2 * y1 + y2), b2 * py - b3 * (2 * z1 + z2)], 1)
        mP = torch.cat([a_ * (x1 - x2), -b2 * pz - b3 * (y1 + 2 * y2), b2 * py - b3 * (z1 + 2 * z2)], 1)
        if prev and bool(lvv.any()):
            dp, d1, d2 = 0.5 * (p2 - s["p2"]), 0.5 * (r1 - s["a1"]), 0.5 * (r2 - s["a2"])
            on = lvv.to(torch.float64) / prev
            gN, gP = on * k["damp"][N], on * k["damp"][P]
            X, Y, Z = (lambda v: v[:, :1]), (lambda v: v[:, 1:2]), (lambda v: v[:, 2:])
            sB1 = k["sA1"]
            pc = torch.cat([k["sA1"] * X(dp), sB1 * Y(dp) - k["sB2"] * (Z(d1) + Z(d2)), sB1 * Z(dp) + k["sB2"] * (Y(d1) + Y(d2))], 1)
            fN, fP = fN + gN * pc, fP - gP * pc
            tw = k["sA2"] * (X(d2) - X(d1))
            mN = mN - 0.5 * gN * torch.cat([-tw, k["sB2"] * Z(dp) + k["sB3"] * (2 * Y(d1) + Y(d2)),
                                            -k["sB2"] * Y(dp) + k["sB3"] * (2 * Z(d1) + Z(d2))], 1)
            mP = mP - 0.5 * gP * torch.cat([tw, k["sB2"] * Z(dp) + k["sB3"] * (Y(d1) + 2 * Y(d2)),
                                            -k["sB2"] * Y(dp) + k["sB3"] * (Z(d1) + 2 * Z(d2))], 1)
        if big:
            fN, mN = _rot(_conj(first), fN), _rot(_conj(first), mN)
        fP, mP = _rot(_conj(e2), fP), _rot(_conj(e2), mP)
        if alive is not None:
            fN, mN, fP, mP = (torch.where(alive, v, torch.zeros_like(v)) for v in (fN, mN, fP, mP))
        force = torch.zeros_like(s["pos"]).index_add(0, N, self.from_x(fN)).index_add(0, P, self.from_x(fP))
        moment = torch.zeros_like(s["pos"]).index_add(0, N, self.from_x(mN)).index_add(0, P, self.from_x(mP))
        # voxels
        m, I = self.mass, self.inertia
        t = _rot(s["q"], force) + self.ext
        if M["gravity"]:
            t = torch.cat([t[:, :2], t[:, 2:] - m * 9.80665 * M["gravity"]], 1)
        if M["contacts"]:
            i, j = self.ci, self.cj
            o = s["pos"][j] - s["pos"][i]
            ln = o.norm(dim=1, keepdim=True)
            over = (0.625 * 2 * L - ln).clamp(min=0)
            stiff = 2 / (1 / k["pen"][i] + 1 / k["pen"][j])
            c = o / ln * (stiff * over)
            t = t.index_add(0, i, -c).index_add(0, j, c)
        static, cur = s["static"], t
        lin = s["lin"]
        if M["floor"]:
            pen = f * L / 2 - L / 2 - s["pos"][:, 2:]
            touch = pen >= 0
            nf = torch.where(touch, k["pen"] * pen, torch.zeros_like(pen))
            slip = static & touch & ((t[:, :2] ** 2).sum(1, True) > (self.mus * nf) ** 2)
            v = lin[:, :2] / m
            l2 = (v * v).sum(1, True)
            sliding = touch & ~static & (l2 > 0)
            l = torch.sqrt(torch.where(sliding, l2, torch.ones_like(l2)))
            fr = torch.where(sliding, -self.muk * nf / l, torch.zeros_like(l)) * v
            cur = torch.cat([t[:, :2] + fr, t[:, 2:] + nf], 1)
            static = static & touch & ~slip
        lin = lin + dt * cur
        move = lin * (dt / m)
        if M["floor"]:
            workd = ((cur - t)[:, :2] * move[:, :2]).sum(1, True)
            ke = 0.5 * (lin[:, :2] ** 2).sum(1, True) / m
            static = touch & (static | (ke + workd <= 0))
            stay = torch.cat([static, static, torch.zeros_like(static)], 1)
            lin, move = lin.masked_fill(stay, 0.0), move.masked_fill(stay, 0.0)
        pos = s["pos"] + move
        ang = s["ang"] + dt * _rot(s["q"], moment)
        q = _qmul(_from_vector(ang * (dt / I)), s["q"])
        if len(self.fixed) or self.ramp is not None:
            zero = torch.zeros_like(pos)
            home = self.x0
            if self.ramp is not None:
                home = home.clone()
                home[self.ramp, 2] += -M["ramp"][1] / dt * s["t"]
            one = torch.zeros_like(q)
            one[:, 0] = 1
            pos, lin = torch.where(self.free, pos, home), torch.where(self.free, lin, zero)
            ang, q = torch.where(self.free, ang, zero), torch.where(self.free, q, one)
        return {"pos": pos, "q": q, "lin": lin, "ang": ang, "static": static, "p2": p2, "a1": r1, "a2": r2, "small": small,
                "lvv": torch.ones_like(lvv) if alive is None else lvv | alive, "strain": strain, "top": top, "off": off,
                "t": s["t"] + dt}

    def transverse(self, s):
        """transverse strain sums and areas of the links, from the strains of the step before"""
        n, L = self.n, self.L
        ext = self.ext != 0
        held = ~self.free
        add, cnt = [], []
        for a, (b, e) in enumerate(self.span):
            st, z = s["strain"][b:e], torch.zeros(n, 1, dtype=torch.float64, device=_dev())
            c = torch.zeros_like(z).index_add(0, self.N[b:e], torch.ones_like(st)).index_add(0, self.P[b:e], torch.ones_like(st))
            v = z.index_add(0, self.N[b:e], st).index_add(0, self.P[b:e], st)
            cnt.append((c == 2) | ((c == 1) & (held | ext[:, a:a + 1])))
            add.append(torch.where(c == 2, 0.5 * v, v))
        r, ten = torch.cat(add, 1), torch.cat(cnt, 1)
        value = (1 + torch.where(ten, r, torch.zeros_like(r)).sum(1, True)) ** (-self.nu) - 1
        r = torch.where(ten, r, value)
        r = torch.where(held, torch.zeros_like(r), r)   # a held voxel keeps the value of the state at rest
        tss, area = [], []
        for a, (b, e) in enumerate(self.span):
            u, w = [r[:, c:c + 1] for c in range(3) if c != a]
            sm, ar = u + w, L * L * (1 + u) * (1 + w)
            i, j = self.N[b:e], self.P[b:e]
            tss.append(0.5 * (sm[i] + sm[j]))
            area.append(0.5 * (ar[i] + ar[j]))
        return torch.cat(tss), torch.cat(area)


def _exact_static(M):
    """conjugate gradients on the assembled beam stiffness, to rounding"""
    X = _Exact(M)
    n, dev = X.n, _dev()
    E, L = X.E0[0].item(), PITCH
    a1, a2, b1, b2, b3 = E * L, E * L ** 3 / 12, E * L, E * L * L / 2, E * L ** 3 / 6
    blocks = []
    for axis, (r1, c1, r2, c2, v) in enumerate(((1, 5, 2, 4, b2), (0, 5, 2, 3, -b2), (0, 4, 1, 3, b2))):
        d = [a1 if axis == j else b1 for j in range(3)]
        K11 = np.diag(d + [a2 if axis == j else 2 * b3 for j in range(3)]).astype(float)
        K22, K12 = K11.copy(), np.diag([-x for x in d] + [-a2 if axis == j else b3 for j in range(3)]).astype(float)
        for K, s in ((K11, v), (K22, -v)):
            K[r1, c1] = K[c1, r1] = s
            K[r2, c2] = K[c2, r2] = -s
        K12[r1, c1], K12[c1, r1], K12[r2, c2], K12[c2, r2] = v, -v, -v, v
        blocks.append([_t(K) for K in (K11, K12, K22)])
    free = X.free.to(torch.float64)
    diag = torch.zeros(n, 6, dtype=torch.float64, device=dev)
    for (b, e), (K11, K12, K22) in zip(X.span, blocks):
        one = torch.ones(e - b, 1, dtype=torch.float64, device=dev)
        diag = diag.index_add(0, X.N[b:e], one * K11.diagonal()).index_add(0, X.P[b:e], one * K22.diagonal())

    def apply(u):
        y = torch.zeros_like(u)
        for (b, e), (K11, K12, K22) in zip(X.span, blocks):
            i, j = X.N[b:e], X.P[b:e]
            y = y.index_add(0, i, u[i] @ K11.T + u[j] @ K12.T).index_add(0, j, u[j] @ K22.T + u[i] @ K12)
        return y * free
    rhs = torch.cat([X.ext, torch.zeros_like(X.ext)], 1) * free
    x = torch.zeros_like(rhs)
    r = rhs.clone()
    z = r / diag * free
    p, rz = z.clone(), (r * z).sum()
    r0 = r.norm()
    for it in range(20000):
        q = apply(p)
        al = rz / (p * q).sum()
        x, r = x + al * p, r - al * q
        if it % 32 == 0 and bool(r.norm() < 1e-14 * r0):
            break
        z = r / diag * free
        new = (r * z).sum()
        p, rz = z + (new / rz) * p, new
    return {"pos": (X.x0 + x[:, :3]).cpu().numpy(), "orient": _from_vector(x[:, 3:]).cpu().numpy()}


def exact(case, seed):
    M = _model(case, seed)
    kind = case["kind"]
    if kind == "static":
        return _exact_static(M)
    X, dt = _Exact(M), M["dt"]
    if kind == "gradient":
        from torch.utils.checkpoint import checkpoint
        log_e = torch.log(_t(M["modulus"])).requires_grad_()
        phase = _t(M["phase"]).requires_grad_()
        s = X.start()

        def one(log_e, phase, s, prev):
            return X.step(s, X.constants(torch.exp(log_e)[:, None]), dt, prev, phase[:, None])
        for i in range(case["steps"]):
            s = checkpoint(one, log_e, phase, s, dt if i else 0.0, use_reentrant=False)
        w = X.mass[:, 0]
        loss, at = 0.0, 0
        for ijk, _ in M["robots"]:
            b = slice(at, at + len(ijk))
            loss = loss - (s["pos"][b, 0] * w[b]).sum() / w[b].sum()
            at += len(ijk)
        loss.backward()
        return {"pos": s["pos"].detach().cpu().numpy(), "d_log_modulus": log_e.grad.cpu().numpy(),
                "d_phase": phase.grad.cpu().numpy()}
    k, s = X.constants(), X.start()
    phase = _t(M["phase"])[:, None] if M["phase"] is not None else None
    with torch.no_grad():
        for i in range(WARM + case["steps"] * case.get("calls", 1)):
            s = X.step(s, k, dt, dt if i else 0.0, phase)
    pos = s["pos"].cpu().numpy()
    if kind == "robots":
        com, at = [], 0
        w = X.mass.cpu().numpy()
        for ijk, _ in M["robots"]:
            b = slice(at, at + len(ijk))
            com.append((pos[b] * w[b]).sum(0) / w[b].sum())
            at += len(ijk)
        return {"com": np.array(com), "pos": pos}
    if case["precision"] == "fp64" and kind in ("beam", "porous") and case.get("calls", 1) == 1:
        return {"pos": pos, "orient": s["q"].cpu().numpy(), "linMom": s["lin"].cpu().numpy(),
                "angMom": s["ang"].cpu().numpy(), "flags": None}
    return {"pos": pos}
