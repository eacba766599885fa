"""Performance cases of the AVBD backend: the frames a user has it simulate.

Every case but the network's is a control interval, the way a trainer, a
robotics loop or a clip renderer drives the solver: put the bodies into a
start state, advance some frames, read the states back -- through
GPUSolver.setBodyStates / submitStep / stepToResidual / bodyStates.  The start
states are contact-rich (a drape on its sphere, a block landing, stacks with
pushed cubes), because that is where a simulation spends its time.  The scene
builders and sizes are those of the package's demos and benchmark.

Scene geometry depends on the case alone and is kept between preparations of
the same case; the states (velocities, jitter) come from the seed.
"""
import functools
import math
import os
import sys

import numpy as np
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
if os.path.join(ROOT, "avbd-metal_amd") not in sys.path:
    sys.path.insert(0, os.path.join(ROOT, "avbd-metal_amd"))

from avbd_amd import GPUSolver, PhysicsScene, SimSettings, WarmStartMLP, demos  # noqa: E402

DT = 1.0 / 60.0


# ---------------------------------------------------------------------------
# cases
# ---------------------------------------------------------------------------
def listed():
    return [
        # one 10-cube stack, the reference's smallest GPU scene: a frame is launch latency
        dict(name="stack_10", kind="stack", bodies=10, frames=8),
        # a small batch of independent rigid scenes (stacks and motor-driven chains), as in a unit test or a small sweep
        dict(name="rigid_batch_64", kind="rigid_batch", scenes=64, frames=4),
        # the benchmark's 4096 uneven rigid scenes in one solver: a training run's environment batch
        dict(name="rigid_batch_4096", kind="rigid_batch", scenes=4096, frames=4),
        # a heap of boxes, spheres and capsules falling into one contact island
        dict(name="pile_300", kind="pile", bodies=300, frames=6),
        # the smallest soft block (smoke-test size), interactive use
        dict(name="block_4", kind="block", cells=4, frames=8, iterations=20),
        # the headline soft block: 9261 vertices, 48000 tets, landing
        dict(name="block_20", kind="block", cells=20, frames=8, iterations=20),
        # the 1M-tet block: memory-bound color sweeps
        dict(name="block_55", kind="block", cells=55, frames=8, iterations=20),
        # a 96^2 sheet folded onto itself: two layers in contact over the whole sheet
        dict(name="cloth_fold_96", kind="cloth", n=96, frames=4, iterations=30, fold=True),
        # the benchmark's 256^2 drape lying on its sphere
        dict(name="cloth_256", kind="cloth", n=256, frames=4, iterations=30, fold=False),
        # 64 uneven soft blocks in one solver (isotropic limiter)
        dict(name="soft_batch_64", kind="soft_batch", scenes=64, frames=4, iterations=20),
        # the other half of the headline metric: frames of the block iterated to residual 1e-4, learned start attached
        dict(name="residual_20", kind="residual", cells=20, frames=2, learned=True),
        # training the warm-start network: one epoch of forward, backward and Adam
        dict(name="mlp_train", kind="mlp_train", rows=65536, batch=4096, outputs=3),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["stack", "rigid_batch", "pile", "block", "cloth", "soft_batch", "residual", "mlp_train"])
    if kind == "stack":
        return dict(kind=kind, bodies=_log_int(rng, 2, 64), frames=rng.randint(1, 8))
    if kind == "rigid_batch":
        return dict(kind=kind, scenes=_log_int(rng, 3, 4000), frames=rng.randint(1, 4))
    if kind == "pile":
        return dict(kind=kind, bodies=_log_int(rng, 20, 1500), frames=rng.randint(1, 6))
    if kind == "block":
        return dict(kind=kind, cells=_log_int(rng, 2, 40), frames=rng.randint(1, 8), iterations=rng.randint(5, 30))
    if kind == "cloth":
        return dict(kind=kind, n=_log_int(rng, 20, 250), frames=rng.randint(1, 4), iterations=rng.randint(8, 30),
                    fold=rng.random() < 0.5)
    if kind == "soft_batch":
        return dict(kind=kind, scenes=_log_int(rng, 2, 64), frames=rng.randint(1, 4), iterations=rng.randint(5, 25))
    if kind == "residual":
        return dict(kind=kind, cells=_log_int(rng, 5, 18), frames=rng.randint(1, 2), learned=rng.random() < 0.5)
    return dict(kind=kind, rows=_log_int(rng, 33, 131072), batch=rng.choice([97, 512, 1024, 4096]),
                outputs=rng.choice([3, 6]))


# ---------------------------------------------------------------------------
# scenes (geometry by the case, kept between preparations)
# ---------------------------------------------------------------------------
def _key(case):
    return tuple(sorted((k, v) for k, v in case.items() if k not in ("name", "frames")))


class _Arrays:
    """The scene's state arrays as bodyStates lays them out."""

    def __init__(self, scene):
        b = scene.bodies
        self.pos = np.array([x["position"] for x in b], np.float32)
        self.rot = np.array([x["rotation"] for x in b], np.float32)
        self.moving = np.array([x["density"] > 0 for x in b])
        self.particle = np.array([x["particle"] for x in b])


@functools.lru_cache(maxsize=2)
def _scene(key):
    c = dict(key)
    kind = c["kind"]
    if kind == "stack":
        s = demos.stack_scene(height=c["bodies"], seed=11)
    elif kind == "rigid_batch":
        s = demos.batched_scene(c["scenes"])[0]
    elif kind == "pile":
        s = _pile(c["bodies"])
    elif kind in ("block", "residual"):
        s = demos.soft_block_scene(cells=c["cells"], bottom=0.02, vel_sigma=0.0, iterations=c.get("iterations", 20))
    elif kind == "soft_batch":
        s = demos.batched_soft_scene(c["scenes"], iterations=c["iterations"])
    else:
        size = 2.0 * (c["n"] - 1) / 255.0
        s = demos.cloth_scene(n=c["n"], size=size, height=0.45 + 0.25 * size + 0.02, radius=2.0e-3, jitter=0.0,
                              sphere_radius=0.25 * size, iterations=c["iterations"])
    return s, _Arrays(s)


def _pile(n):
    """Boxes, spheres and capsules of 0.24 to 0.34 m stacked on a jittered
    lattice 9 columns wide: a heap settling on the ground."""
    s = PhysicsScene("pile", SimSettings(iterations=10))
    demos.add_ground(s)
    rng = demos.SplitMix64(77)
    for i in range(n):
        x, y, z = (i % 9 - 4) * 0.35, (i // 9 % 9 - 4) * 0.35, 0.18 + 0.33 * (i // 81)
        p = (x + rng.uniform(-0.01, 0.01), y + rng.uniform(-0.01, 0.01), z)
        k = rng.next() % 3
        if k == 0:
            s.addBody(tuple(rng.uniform(0.24, 0.34) for _ in range(3)), 1.0, 0.5, p)
        elif k == 1:
            s.addSphere(rng.uniform(0.24, 0.34), 1.0, 0.5, p)
        else:
            s.addCapsule(rng.uniform(0.06, 0.1), rng.uniform(0.1, 0.12), 1.0, 0.5, p)
    return s


def _start(case, seed):
    """(scene, pos, rot, vel, angvel): the start state of the interval."""
    scene, a = _scene(_key(case))
    rng = np.random.default_rng(seed)
    n = len(a.pos)
    pos, rot = a.pos.copy(), a.rot.copy()
    vel, ang = np.zeros((n, 3), np.float32), np.zeros((n, 3), np.float32)
    kind, m = case["kind"], a.moving
    if kind in ("stack", "rigid_batch", "pile"):
        # pushed bodies: what a disturbance or an action leaves behind
        vel[m] = rng.normal(0.0, 0.2, (int(m.sum()), 3))
        ang[m] = rng.normal(0.0, 0.2, (int(m.sum()), 3))
        if kind == "pile":
            vel[m, 2] -= 1.0
    elif kind in ("block", "residual", "soft_batch"):
        # landing, with the benchmark's velocity noise (less on finer lattices: particles of one block stay apart)
        sigma = 0.1 if kind == "soft_batch" else min(0.1, 2.0 / case["cells"])
        vel[m] = rng.normal(0.0, sigma, (int(m.sum()), 3))
        vel[m, 2] -= 1.0
    else:
        size = 2.0 * (case["n"] - 1) / 255.0
        pos[m] = _folded(pos[m], case["n"], rng) if case["fold"] else _draped(pos[m], 0.25 * size, rng)
        vel[m] = rng.normal(0.0, 0.01, (int(m.sum()), 3))
        vel[m, 2] -= 0.2
    return scene, pos, rot, vel, ang


def _draped(p, radius, rng):
    """The flat sheet laid over the sphere (centre z 0.45): along each radius
    onto the sphere up to 0.6 rad, then straight off it; 0.1 mm of noise."""
    s = np.hypot(p[:, 0].astype(np.float64), p[:, 1])
    rg = radius + 3.0e-3
    phi = np.minimum(s / rg, 0.6)
    rest = np.maximum(s - 0.6 * rg, 0.0)
    r = rg * np.sin(phi) + rest * np.cos(phi)
    z = 0.45 + rg * np.cos(phi) - rest * np.sin(phi)
    k = r / np.maximum(s, 1e-12)
    out = np.stack([p[:, 0] * k, p[:, 1] * k, z], 1)
    return (out + rng.uniform(-1e-4, 1e-4, out.shape)).astype(np.float32)


def _folded(p, n, rng):
    """The flat sheet folded at its middle column, the second half 4.2 mm over
    the first (the particles' radii sum to 4 mm), dropping onto the sphere."""
    g = p.astype(np.float64).reshape(n, n, 3)
    half = n // 2
    ym = 0.5 * (g[:, half - 1, 1] + g[:, half, 1])
    g[:, half:, 1] = 2.0 * ym[:, None] - g[:, half:, 1]
    g[:, half:, 2] += 4.2e-3
    out = g.reshape(-1, 3)
    return (out + rng.uniform(-1e-4, 1e-4, out.shape)).astype(np.float32)


# ---------------------------------------------------------------------------
# prepare / run
# ---------------------------------------------------------------------------
def _mlp_data(case, seed):
    """Feature rows and targets of the magnitudes that the solver's own
    samples have, and starting parameters."""
    rng = np.random.default_rng(seed)
    x = rng.normal(0.0, 0.5, (case["rows"], 24)).astype(np.float32)
    w = rng.normal(0.0, 0.4, (24, case["outputs"]))
    t = (np.tanh(x @ w) + 0.1 * rng.normal(0.0, 1.0, (case["rows"], case["outputs"]))).astype(np.float32)
    p = []
    for fan_in, shape in ((24, (24, 128)), (0, (128,)), (128, (128, 128)), (0, (128,)), (128, (128, case["outputs"])),
                          (0, (case["outputs"],))):
        p.append((rng.uniform(-1.0, 1.0, shape) / math.sqrt(fan_in) if fan_in else np.zeros(shape)).reshape(-1))
    return x, t, np.concatenate(p).astype(np.float32)


def prepare(case, seed):
    if case["kind"] == "mlp_train":
        x, t, p = _mlp_data(case, seed)
        return dict(kind="mlp_train", net=WarmStartMLP(seed=1, outputs=case["outputs"]), x=x, t=t, params=p,
                    batch=case["batch"])
    scene, pos, rot, vel, ang = _start(case, seed)
    solver = GPUSolver(scene)
    idx = np.arange(len(pos), dtype=np.uint32)
    state = dict(kind=case["kind"], solver=solver, frames=case["frames"], start=(idx, pos, rot, vel, ang))
    if case.get("learned"):
        state["net"] = WarmStartMLP(seed=3)
        solver.setWarmStart(state["net"], smooth=2)
    return state


def run(state):
    if state["kind"] == "mlp_train":
        net = state["net"]
        net.params = state["params"]
        losses = net.train(state["x"], state["t"], epochs=1, batch=state["batch"], lr=1e-3, seed=5)
        return net.params, losses
    solver = state["solver"]
    solver.setBodyStates(*state["start"])
    for _ in range(state["frames"]):
        if state["kind"] == "residual":
            solver.stepToResidual(1e-4, 1000, 10)
        else:
            solver.submitStep()
    return solver.bodyStates()


# ---------------------------------------------------------------------------
# work and tolerance
# ---------------------------------------------------------------------------
def work(case):
    """Bytes: per frame every body's state (52 B) in and out and each element
    or joint record once; flops: per sweep the element, contact and block
    solve arithmetic of the dynamic bodies."""
    if case["kind"] == "mlp_train":
        o, r = case["outputs"], case["rows"]
        return {"bytes": 4.0 * r * (24 + o), "flops": 3.0 * 2.0 * r * (24 * 128 + 128 * 128 + 128 * o)}
    scene, a = _scene(_key(case))
    nb, nd = len(a.pos), int(a.moving.sum())
    tets, tris, springs, joints = len(scene.tets), len(scene.tris), len(scene.springs), len(scene.joints)
    sweeps = 200 if case["kind"] == "residual" else scene.settings.iterations
    rigid = int((a.moving & ~a.particle).sum())
    per_sweep = (4 * 150.0 * tets + 3 * 120.0 * tris + 2 * 40.0 * springs + 4 * 40.0 * tris + 2 * 400.0 * joints
                 + 4 * 2 * 200.0 * rigid + 250.0 * rigid + 60.0 * (nd - rigid))
    per_frame = 2 * 52.0 * nb + 60.0 * tets + 60.0 * tris + 32.0 * springs + 224.0 * joints
    return {"bytes": case["frames"] * per_frame, "flops": case["frames"] * sweeps * per_sweep}


def tolerance(case):
    """About four times what a pass moves when a body's sums are taken over
    another number of lanes; velocities are position differences times 60,
    and a disturbed rigid scene amplifies rounding (the measured worst:
    stack and batches 5e-4, sheets 3e-5, blocks 6e-6).  The network: bf16
    operands through an epoch of Adam, 2e-3 off 64 bits."""
    return {"stack": {"rel": 2e-3, "max": 0.05}, "rigid_batch": {"rel": 2e-3, "max": 0.5},
            "pile": {"rel": 2e-3, "max": 0.5}, "cloth": {"rel": 1e-4, "max": 2e-3},
            "block": {"rel": 2.5e-5, "max": 5e-4}, "soft_batch": {"rel": 2.5e-5, "max": 5e-4},
            "residual": {"rel": 5e-5, "max": 1e-3}, "mlp_train": {"rel": 8e-3, "max": 0.3}}[case["kind"]]


# ---------------------------------------------------------------------------
# 64-bit references: soft blocks (Stable Neo-Hookean tets on a ground plane)
# and the network
# ---------------------------------------------------------------------------
def exact(case, seed):
    if case["kind"] == "mlp_train":
        return _exact_train(case, seed)
    if case["kind"] not in ("block", "residual", "soft_batch"):
        return None  # contact sets of rigid shapes and sheets: minutes in plain torch
    scene, pos, rot, vel, ang = _start(case, seed)
    ref = _SoftReference(_key(case), scene, pos, vel)
    for _ in range(case["frames"]):
        ref.frame(scene.settings.iterations, 1e-4 if case["kind"] == "residual" else None)
    return ref.x.cpu().numpy(), rot.astype(np.float64), ref.v.cpu().numpy(), np.zeros((len(pos), 3))


@functools.lru_cache(maxsize=1)
def _soft_topology(key):
    """Greedy colors (index order, lowest color unused by a lower neighbour)
    and per color the tets of each vertex with the vertex's own corner first."""
    scene, a = _scene(key)
    tets = np.array([t[0] for t in scene.tets], np.int64)
    mat = np.array([t[1:] for t in scene.tets], np.float32)
    n = len(a.pos)
    lower = np.concatenate([tets[:, [i, j]] for i in range(4) for j in range(4) if i != j])
    lower = np.unique(lower[lower[:, 0] > lower[:, 1]], axis=0)
    first = np.searchsorted(lower[:, 0], np.arange(n + 1))
    nbr = lower[:, 1].tolist()
    color = [0] * n
    for v in range(n):
        used = {color[u] for u in nbr[first[v]:first[v + 1]]}
        c = 0
        while c in used:
            c += 1
        color[v] = c
    color = np.array(color)
    x = a.pos.astype(np.float64)
    d = np.stack([x[tets[:, k]] - x[tets[:, 0]] for k in (1, 2, 3)], 2)
    inv, vol = np.linalg.inv(d), np.abs(np.linalg.det(d)) / 6.0
    own = tets.reshape(-1)
    order = np.argsort(own, kind="stable")
    start = np.searchsorted(own[order], np.arange(n + 1))
    deg = np.diff(start)
    groups = []
    for c in range(color.max() + 1):
        bodies = np.nonzero((color == c) & a.moving & (deg > 0))[0]
        k = int(deg[bodies].max()) if len(bodies) else 0
        slot = start[bodies][:, None] + np.arange(k)[None, :]
        valid = np.arange(k)[None, :] < deg[bodies][:, None]
        e = order[np.where(valid, slot, 0)]
        groups.append((bodies, e // 4, e % 4, valid))
    return tets, mat, inv, vol, groups


class _SoftReference:
    def __init__(self, key, scene, pos, vel):
        dev = "cuda" if torch.cuda.is_available() else "cpu"
        tets, mat, inv, vol, groups = _soft_topology(key)
        f8 = functools.partial(torch.as_tensor, dtype=torch.float64, device=dev)
        i8 = functools.partial(torch.as_tensor, dtype=torch.int64, device=dev)
        self.tets, self.inv = i8(tets), f8(inv)
        self.mu = f8((mat[:, 0].astype(np.float64) * vol))
        self.lam = f8((mat[:, 1].astype(np.float64) * vol))
        self.groups = []
        for bodies, t, corner, valid in groups:
            if not len(bodies):
                continue
            w = np.concatenate([-inv.sum(1, keepdims=True), inv], 1)  # shape-function gradients of the 4 corners
            self.groups.append((i8(bodies), i8(t), f8(w)[i8(t), i8(corner)], f8(valid)))
        b = scene.bodies
        self.r = f8(np.array([x["size"][0] * 0.5 for x in b]))
        vol_s = 4.0 / 3.0 * math.pi * self.r ** 3
        part = f8(np.array([float(x["particle"]) for x in b]))
        self.m = f8(np.array([x["density"] for x in b], np.float32)) * vol_s * part
        self.dyn = self.m > 0
        fr = f8(np.array([x["friction"] for x in b], np.float32))
        self.mu_c = torch.sqrt(fr * fr[0])
        self.set = scene.settings
        self.x, self.v, self.vp = f8(pos), f8(vel), f8(vel)
        n = len(pos)
        z3 = f8(np.zeros((n, 3)))
        self.pen, self.lm, self.anchor = z3.clone(), z3.clone(), z3[:, :2].clone()
        self.stick = torch.zeros(n, dtype=torch.bool, device=dev)
        self.had = torch.zeros(n, dtype=torch.bool, device=dev)

    def elastic(self, x, g):
        """Gradient and Hessian block of group g's vertices: SNH per tet,
        energy mu/2 (Ic - 3) + lambda/2 (J - 1 - mu/lambda)^2."""
        bodies, t, w, valid = g
        p = x[self.tets[t]]
        d = p[:, :, 1:] - p[:, :, :1]
        f = torch.einsum("nkei,nkej->nkij", d, self.inv[t])  # F = sum_e d_e (row e of Dm^-1)
        f0, f1, f2 = f[..., 0], f[..., 1], f[..., 2]
        j0, j1, j2 = torch.linalg.cross(f1, f2), torch.linalg.cross(f2, f0), torch.linalg.cross(f0, f1)
        mu, lam = self.mu[t], self.lam[t]
        s = lam * ((f0 * j0).sum(-1) - 1.0 - mu / lam)
        gj = j0 * w[..., :1] + j1 * w[..., 1:2] + j2 * w[..., 2:]
        fw = f0 * w[..., :1] + f1 * w[..., 1:2] + f2 * w[..., 2:]
        grad = ((fw * mu[..., None] + gj * s[..., None]) * valid[..., None]).sum(1)
        h = torch.einsum("nk,nki,nkj->nij", lam * valid, gj, gj)
        diag = (mu * (w * w).sum(-1) * valid).sum(1)
        return grad, h + diag[:, None, None] * torch.eye(3, dtype=torch.float64, device=x.device)

    def contact(self, x):
        """C, F and the friction bound of every particle's ground contact
        (normal -z from the ground's side, tangents y and x)."""
        dq = x - self.x0
        d = torch.stack([dq[:, 2], -dq[:, 1], -dq[:, 0]], 1)
        c = self.c0 * (1.0 - self.set.alpha) + d
        f = self.pen * c + self.lm
        f[:, 0].clamp_(max=0.0)
        bound = f[:, 0].abs() * self.mu_c
        fs = torch.hypot(f[:, 1], f[:, 2])
        k = torch.where((fs > bound) & (fs > 0), bound / fs.clamp(min=1e-300), torch.ones_like(fs))
        return c, torch.stack([f[:, 0], f[:, 1] * k, f[:, 2] * k], 1), fs, bound

    def gradient(self, x, g):
        b = g[0]
        grad, h = self.elastic(x, g)
        md = self.m[b] / DT32 ** 2
        grad = grad + (x[b] - self.inert[b]) * md[:, None]
        _, f, _, _ = self.contact(x)
        on = self.on[b].double()[:, None]
        f, k = f[b] * on, self.pen[b] * on
        # rows of the particle's side: -n = +z, -t1 = -y, -t2 = -x
        grad = grad + torch.stack([-f[:, 2], -f[:, 1], f[:, 0]], 1)
        return grad, h + torch.diag_embed(md[:, None] + torch.stack([k[:, 2], k[:, 1], k[:, 0]], 1))

    def sweep(self):
        s = self.set
        for g in self.groups:
            b = g[0]
            grad, h = self.gradient(self.x, g)
            dx = -torch.linalg.solve(h, grad)
            lim = 0.35 * self.r[b]
            ln = dx.norm(dim=1)
            self.x[b] += dx * torch.where(ln > lim, lim / ln.clamp(min=1e-300), torch.ones_like(ln))[:, None]
        c, f, fs, bound = self.contact(self.x)
        f[:, 0] = torch.maximum(f[:, 0], -torch.clamp(1.0e5 * self.m, min=10.0).clamp(max=s.lambdaMax))
        self.lm = torch.where(self.on[:, None], f, self.lm)
        push = self.on & (f[:, 0] < 0)
        self.pen[:, 0] = torch.where(push, (self.pen[:, 0] + s.betaLin * c[:, 0].abs()).clamp(max=1e10), self.pen[:, 0])
        hold = self.on & (fs <= bound)
        for k in (1, 2):
            self.pen[:, k] = torch.where(hold, (self.pen[:, k] + s.betaLin * c[:, k].abs()).clamp(max=1e6),
                                         self.pen[:, k])
        self.stick = torch.where(hold, torch.hypot(c[:, 1], c[:, 2]) < 1e-5, self.stick)

    def residual(self):
        g2 = sum(float((self.gradient(self.x, g)[0] ** 2).sum()) for g in self.groups)
        return math.sqrt(g2 / float(((self.m * self.set.gravity) ** 2).sum()))

    def frame(self, iterations, tol):
        s, x, v = self.set, self.x, self.v
        # ground contacts (top face z = 0) within the margin plus the approach of one step
        reach = torch.minimum((-v[:, 2]).clamp(min=0.0) * DT32,
                              torch.clamp(3.0 * self.r, min=4.0 * s.collisionMargin).clamp(max=0.25))
        self.on = self.dyn & (x[:, 2] <= self.r + s.collisionMargin + reach)
        kept = self.on & self.had
        self.anchor = torch.where((kept & self.stick)[:, None], self.anchor, x[:, :2])
        d = torch.stack([self.anchor[:, 0] - x[:, 0], self.anchor[:, 1] - x[:, 1], self.r - x[:, 2]], 1)
        self.c0 = torch.stack([-d[:, 2] + s.collisionMargin, d[:, 1], d[:, 0]], 1)
        floor = torch.clamp(self.m / DT32 ** 2, min=1.0, max=1e10)
        lo = torch.stack([floor, floor.clamp(max=1e6), floor.clamp(max=1e6)], 1)
        self.lm = torch.where(kept[:, None], self.lm * (s.alpha * s.gamma), torch.zeros_like(self.lm))
        self.pen = torch.maximum(torch.where(kept[:, None], self.pen * s.gamma, torch.zeros_like(self.pen)), lo)
        self.stick = self.stick & kept
        # inertial target and adaptive guess
        dyn = self.dyn[:, None]
        gz = torch.zeros_like(x)
        gz[:, 2] = s.gravity
        self.x0 = x.clone()
        self.inert = x + v * DT32 + gz * DT32 ** 2
        w = (((v - self.vp)[:, 2] / DT32) / s.gravity).clamp(0.0, 1.0)[:, None]
        self.x = torch.where(dyn, x + v * DT32 + gz * (w * DT32 ** 2), x)
        if tol is None:
            for _ in range(iterations):
                self.sweep()
        else:
            for _ in range(100):
                for _ in range(10):
                    self.sweep()
                if self.residual() <= tol:
                    break
        self.had = self.on
        self.vp = v
        self.v = torch.where(dyn, (self.x - self.x0) / DT32, v)


DT32 = float(np.float32(DT))


def _splitmix(state):
    m = (1 << 64) - 1
    state = (state + 0x9E3779B97F4A7C15) & m
    z = state
    z = ((z ^ (z >> 30)) * 0xBF58476D1CE4E5B9) & m
    z = ((z ^ (z >> 27)) * 0x94D049BB133111EB) & m
    return state, z ^ (z >> 31)


def _exact_train(case, seed):
    """One epoch of Adam on shuffled batches in 64 bits."""
    x, t, p = _mlp_data(case, seed)
    o, n = case["outputs"], case["rows"]
    order, st = list(range(n)), 5
    for i in range(n - 1, 0, -1):
        st, z = _splitmix(st)
        j = z % (i + 1)
        order[i], order[j] = order[j], order[i]
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    x, t = torch.as_tensor(x, device=dev).double(), torch.as_tensor(t, device=dev).double()
    p = torch.as_tensor(p, device=dev).double()
    order = torch.as_tensor(order, device=dev)
    sizes = [24 * 128, 128, 128 * 128, 128, 128 * o, o]
    m, v, losses = torch.zeros_like(p), torch.zeros_like(p), []
    b = min(case["batch"], n)
    for k in range(max(1, n // b)):
        rows = order[k * b:(k + 1) * b]
        q = p.clone().requires_grad_(True)
        w1, b1, w2, b2, w3, b3 = torch.split(q, sizes)
        h = torch.relu(torch.addmm(b1, x[rows], w1.view(24, 128)))
        h = torch.relu(torch.addmm(b2, h, w2.view(128, 128)))
        loss = ((torch.addmm(b3, h, w3.view(128, o)) - t[rows]) ** 2).mean()
        g, = torch.autograd.grad(loss, q)
        losses.append(float(loss.detach()))
        m, v = 0.9 * m + 0.1 * g, 0.999 * v + 0.001 * g * g
        p = p - 1e-3 * (m / (1 - 0.9 ** (k + 1))) / (torch.sqrt(v / (1 - 0.999 ** (k + 1))) + 1e-8)
    return p.cpu().numpy(), np.array([sum(losses) / len(losses)])
