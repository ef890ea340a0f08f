"""The work that users of flipsolver2d_amd have it do, as cases that a harness can time and compare.

Two families:

  solve   LinearSolver::solve on the GPU: one pressure system in host memory (materials, right-hand side) in, the
          pressure out (`Context.poisson_solve`).
  scenes  simulations: first-frame set-up from polygons, a few frames, and the state that a caller reads back (the
          particles, the velocity grid, the materials and the level sets: what the C++ API's accessors fetch).  One scene
          alone, one scene stepped through the stage hooks, a batch, or requests to a server.

`listed()` names the cases, `draw(rng)` gives more of the same ranges.  `prepare` makes what a program holds before the
call, `run` is one pass, `work` what a pass cannot do without and `exact` the pressure in 64 bits.
"""
import ctypes
import math

import numpy as np
import torch

import flipsolver2d_amd as fg

TOL = 1e-6          # relative residual of every pressure solve
PCG_LIMIT = 4000


def listed():
    return [
        # a small scene's pressure system in a tight loop that may not allocate: launches and host round trips
        {"name": "solve_64_noalloc", "kind": "solve", "I": 64, "J": 64, "mask": "dam", "noalloc": True},
        # a caller's own solver on a ragged grid, porous liquid
        {"name": "solve_517x333", "kind": "solve", "I": 517, "J": 333, "mask": "noise", "noalloc": False},
        # the largest isolated projection: ~60 % liquid, 2 % random solids
        {"name": "solve_4096", "kind": "solve", "I": 4096, "J": 4096, "mask": "noise", "noalloc": False},
        # an interactive preview: the smallest scene, latency alone
        {"name": "dam_64", "kind": "scene", "solver": "flip", "I": 64, "J": 64, "ppc": 4, "frames": 3, "setup": "dam"},
        # the plain dam break at its usual resolution
        {"name": "dam_128", "kind": "scene", "solver": "flip", "I": 128, "J": 128, "ppc": 4, "frames": 4, "setup": "dam"},
        # the same at production resolution: 2.3 M particles
        {"name": "dam_1024", "kind": "scene", "solver": "flip", "I": 1024, "J": 1024, "ppc": 8, "frames": 3, "setup": "dam"},
        # a scene file's objects (friction, source, sink) on a grid with no round side
        {"name": "sources_225x150", "kind": "scene", "solver": "flip", "I": 225, "J": 150, "ppc": 4, "frames": 5,
         "setup": "fountain"},
        # a subclass that overrides a stage hook: step() runs stage by stage
        {"name": "hooks_160x96", "kind": "hooks", "solver": "flip", "I": 160, "J": 96, "ppc": 6, "frames": 3, "setup": "dam"},
        # narrow-band FLIP at production resolution: grids and level sets, few particles
        {"name": "nbflip_1024", "kind": "scene", "solver": "nbflip", "I": 1024, "J": 1024, "ppc": 8, "frames": 3,
         "setup": "dam"},
        # viscous liquids stepped together: the FP64 viscosity solve and a second projection a substep
        {"name": "viscous_8x256", "kind": "batch", "solver": "viscous", "count": 8, "lo": 256, "hi": 256, "lanes": 1,
         "frames": 3},
        # many scenes of uneven size at once, four lanes (what the lane autotuner settles on)
        {"name": "batch_64_mixed", "kind": "batch", "solver": "flip", "count": 64, "lo": 64, "hi": 256, "lanes": 4,
         "frames": 3},
        # requests of uneven size and length served by continuous batching
        {"name": "served_24", "kind": "serve", "count": 24, "lo": 64, "hi": 512, "frames": 4},
    ]


def _side(rng, lo, hi):
    """A side log-uniform in [lo, hi], even or odd."""
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["solve", "solve", "scene", "scene", "scene", "hooks", "batch", "serve"])
    if kind == "solve":
        noalloc = rng.random() < 0.3
        hi = 640 if noalloc else 3200
        return {"kind": "solve", "I": _side(rng, 48, hi), "J": _side(rng, 48, hi),
                "mask": rng.choice(["dam", "noise"]), "noalloc": noalloc}
    if kind == "batch":
        solver = rng.choice(["flip", "flip", "nbflip", "viscous"])
        lo = _side(rng, 48, 128)
        return {"kind": "batch", "solver": solver, "count": rng.randint(3, 8 if solver == "viscous" else 40), "lo": lo,
                "hi": min(256, _side(rng, lo, 320)), "lanes": rng.randint(1, 4), "frames": rng.randint(2, 3)}
    if kind == "serve":
        return {"kind": "serve", "count": rng.randint(4, 20), "lo": _side(rng, 48, 100), "hi": _side(rng, 128, 480),
                "frames": rng.randint(2, 4)}
    solver = "flip" if kind == "hooks" else rng.choice(["flip", "flip", "nbflip", "viscous"])
    hi = 256 if kind == "hooks" or solver == "viscous" else 900
    I = _side(rng, 48, hi)
    J = min(hi, max(48, int(I * rng.uniform(0.6, 1.6))))
    return {"kind": kind, "solver": solver, "I": I, "J": J, "ppc": rng.randint(4, 8), "frames": rng.randint(2, 3),
            "setup": rng.choice(["dam", "fountain"]) if solver == "flip" else "dam"}


# ---------------------------------------------------------------------------------------------------------------------
# pressure systems
# ---------------------------------------------------------------------------------------------------------------------
def _smooth(x, sigma):
    """Gaussian smoothing of a 2-D tensor, reflecting edges, as two passes of shifted sums."""
    radius = int(4 * sigma)
    w = torch.exp(-0.5 * (torch.arange(-radius, radius + 1, dtype=torch.float64) / sigma) ** 2)
    w = (w / w.sum()).tolist()
    for dim in (0, 1):
        n = x.shape[dim]
        at = torch.arange(-radius, n + radius, device=x.device)
        at = at.remainder(2 * n)
        ext = x.index_select(dim, torch.where(at < n, at, 2 * n - 1 - at))
        x = sum(w[k] * ext.narrow(dim, k, n) for k in range(2 * radius + 1))
    return x


def _system(case, seed):
    """(material, right-hand side, scale) on the GPU.  "noise": Gaussian-smoothed uniform noise cut at its 40th
    percentile, 2 % solid cells, face velocities uniform in [-1, 1] (the isolated projection); "dam": the dam break's
    rectangle, a slumping flow and noise.  Both inside a one-cell solid border."""
    I, J = case["I"], case["J"]
    g = torch.Generator(device="cuda").manual_seed(seed)
    rand = lambda *shape: torch.rand(*shape, generator=g, device="cuda")  # noqa: E731
    mat = torch.full((I, J), fg.EMPTY, dtype=torch.int8, device="cuda")
    u, v = 2 * rand(I + 1, J) - 1, 2 * rand(I, J + 1) - 1
    if case["mask"] == "noise":
        field = _smooth(rand(I, J), 8.0)
        mat[field > field.flatten().kthvalue(max(1, int(0.4 * I * J))).values] = fg.FLUID
        solid = rand(I, J) < 0.02
    else:
        mat[int(0.3 * I):, : int(0.4 * J)] = fg.FLUID
        solid = torch.zeros(I, J, dtype=torch.bool, device="cuda")
        x = torch.linspace(0, 1, I + 1, device="cuda")[:, None]
        y = torch.linspace(0, 1, J + 1, device="cuda")[None, :]
        u = 0.1 * u + 0.3 * (1 - x) * torch.cos(3 * y[:, :J])
        v = 0.1 * v + 0.3 * x[:I] * torch.sin(2 * y)
    solid[0], solid[-1], solid[:, 0], solid[:, -1] = True, True, True, True
    mat[solid] = fg.SOLID
    dx = 1.0 / max(I, J)
    s = torch.nn.functional.pad(solid, (1, 1, 1, 1), value=True).double()
    u0, u1, v0, v1 = u[:-1], u[1:], v[:, :-1], v[:, 1:]
    b = -(((u1 - u0) + v1) - v0).double()
    b += (-s[:-2, 1:-1] * u0 + s[2:, 1:-1] * u1 - s[1:-1, :-2] * v0 + s[1:-1, 2:] * v1)
    b = torch.where(mat == fg.FLUID, b / dx, torch.zeros_like(b))
    return mat, b, (1.0 / 30) / (1000.0 * dx * dx)


def exact(case, seed):
    """The pressure by Jacobi-preconditioned conjugate gradients in 64 bits, far past the tolerance of the path.  A
    simulation's frames have no such value."""
    if case["kind"] != "solve":
        return None
    mat, b, scale = _system(case, seed)
    fluid = torch.nn.functional.pad(mat == fg.FLUID, (1, 1, 1, 1)).double()
    open_ = torch.nn.functional.pad(mat != fg.SOLID, (1, 1, 1, 1)).double()
    on = fluid[1:-1, 1:-1]
    n = open_[:-2, 1:-1] + open_[2:, 1:-1] + open_[1:-1, :-2] + open_[1:-1, 2:]
    inv = torch.where((on > 0) & (n > 0), 1 / n.clamp(min=1), torch.zeros_like(n))

    def apply(p):
        e = torch.nn.functional.pad(p, (1, 1, 1, 1))
        return on * (n * p - e[:-2, 1:-1] - e[2:, 1:-1] - e[1:-1, :-2] - e[1:-1, 2:])

    r = b / scale * on
    x, z = torch.zeros_like(r), inv * r
    p, rz, stop = z.clone(), (r * z).sum(), 1e-14 * float(r.norm())
    for k in range(12000):
        q = apply(p)
        alpha = rz / (p * q).sum()
        x += alpha * p
        r -= alpha * q
        if k % 50 == 49 and float(r.norm()) <= stop:
            break
        z = inv * r
        rz, old = (r * z).sum(), rz
        p = z + (rz / old) * p
    return {"pressure": x.flatten()}


# ---------------------------------------------------------------------------------------------------------------------
# scenes
# ---------------------------------------------------------------------------------------------------------------------
def _objects(case, seed):
    """init_objects' arguments: a dam break, or a box with a leaning obstacle, a source, a sink and a pool."""
    I, J = case["I"], case["J"]
    dx = 1.0 / max(I, J)
    h, w = I * dx, J * dx
    walls = [fg.box(0, dx, 0, w), fg.box(h - dx, h, 0, w), fg.box(0, h, 0, dx), fg.box(0, h, w - dx, w)]
    rect = lambda x0, x1, y0, y1: fg.box(max(x0 * h, dx), min(x1 * h, h - dx), max(y0 * w, dx), min(y1 * w, w - dx))  # noqa: E731
    if case["setup"] == "dam":
        o = {"solids": walls, "fluids": [rect(*case.get("box", (0.3, 1.0, 0.0, 0.4)))], "friction": np.zeros(4, np.float32)}
        if case["solver"] == "viscous":
            o["fluid_viscosity"] = [10.0]
    else:
        lean = np.array([[0.55 * h, 0.35 * w], [0.8 * h, 0.45 * w], [0.8 * h, 0.55 * w], [0.55 * h, 0.45 * w]], np.float32)
        o = {"solids": walls + [lean], "friction": np.array([0, 0, 0, 0, 0.3], np.float32),
             "sources": [rect(0.1, 0.2, 0.15, 0.3)], "emitters": [(1.0, 0.5, True)],
             "sinks": [rect(0.85, 1.0, 0.85, 1.0)], "fluids": [rect(0.6, 1.0, 0.0, 0.3)]}
    return dict(o, seed=seed)


def _params(case):
    g = case.get("gravity", (9.81, 0.0))
    return fg.make_params(case["I"], case["J"], ppc=case["ppc"], tol=TOL, pcg_iter_limit=PCG_LIMIT, gravity=g,
                          sim=fg.SIM_NBFLIP if case["solver"] == "nbflip" else fg.SIM_FLIP,
                          viscosity=case["solver"] == "viscous")


def _members(case):
    """The scenes of a batch or of a request stream: sizes and fluid rectangles fixed by the case, as scene dicts."""
    rng = np.random.default_rng(case["count"] * 1000 + case["lo"] + case["hi"])
    out = []
    for _ in range(case["count"]):
        if case["kind"] == "serve":
            n = int(round(np.exp(rng.uniform(np.log(case["lo"]), np.log(case["hi"])))))
        else:
            n = int(rng.choice([max(case["lo"], min(case["hi"], r)) for r in fg.MIXED_RESOLUTIONS]))
        x, y = np.sort(rng.uniform(0.1, 0.6, 2)), np.sort(rng.uniform(0.1, 0.6, 2))
        solver = case.get("solver", "flip")
        box, ppc = (float(x[0]), float(x[1]), float(y[0]), float(y[1])), int(rng.integers(4, 9))
        if solver == "viscous":
            top = rng.uniform(0.4, 0.9)
            box, ppc = (top - rng.uniform(0.2, 0.4), top, 0.0, rng.uniform(0.25, 0.6)), 8
        frames = int(rng.integers(1, case["frames"] + 1)) if case["kind"] == "serve" else case["frames"]
        out.append({"solver": solver, "I": n, "J": n, "ppc": ppc, "setup": "dam", "box": box, "frames": frames})
    return out


class _Reader:
    """The arrays a caller keeps for what it reads after the last frame (the C++ API's sync() fetches these): one array a
    quantity for all its scenes, a stretch of it each.  Particles fill the front of their stretch, `particles` says how far."""

    PARTICLE = {"px": np.float32, "py": np.float32, "vx": np.float32, "vy": np.float32, "pid": np.uint32}
    GRID = {"u": (np.float32, 1, 0), "v": (np.float32, 0, 1), "u_valid": (np.uint8, 1, 0), "v_valid": (np.uint8, 0, 1),
            "material": (np.int8, 0, 0), "fluid_sdf": (np.float32, 0, 0), "solid_sdf": (np.float32, 0, 0)}

    def __init__(self, params):
        size = {k: [p.max_particles for p in params] for k in self.PARTICLE}
        size.update({k: [(p.size_i + di) * (p.size_j + dj) for p in params] for k, (_, di, dj) in self.GRID.items()})
        self.out = {k: np.zeros(sum(size[k]), t) for k, t in self.PARTICLE.items()}
        self.out.update({k: np.zeros(sum(size[k]), t) for k, (t, _, _) in self.GRID.items()})
        self.out["particles"] = np.zeros(len(params), np.int64)
        self.states = []
        for at in range(len(params)):
            state = fg.SceneState()
            for k, n in size.items():
                setattr(state, k, self.out[k][sum(n[:at]):].ctypes.data)
            self.states.append(state)

    def read(self, scenes):
        for at, (scene, state) in enumerate(zip(scenes, self.states)):
            fg._check(fg.lib().fg_scene_get_state(scene.h, ctypes.byref(state)))
            self.out["particles"][at] = state.n_particles
        return self.out


class _Simulation:
    """The context, scenes and read-back arrays of one scene case."""

    def __init__(self, case, seed):
        rng = np.random.default_rng(seed)
        self.case, self.ctx, self.scenes, self.server = case, fg.Context(0), [], None
        members = [case] if case["kind"] in ("scene", "hooks") else _members(case)
        angles = np.deg2rad(rng.uniform(-30.0, 30.0, len(members)))
        seeds = rng.integers(1, 2**31 - 1, len(members))
        if len(members) > 1 or case["kind"] in ("batch", "serve"):
            members = [dict(m, gravity=(9.81 * math.cos(a), 9.81 * math.sin(a))) for m, a in zip(members, angles)]
        self.members = [(m, _params(m), _objects(m, int(s))) for m, s in zip(members, seeds)]
        self.reader = _Reader([p for _, p, _ in self.members])
        if case["kind"] == "serve":
            self.server = fg.Server(self.ctx, hbm_budget=200 << 30, max_resident=256)
        else:
            self.ctx.set_batch_lanes(case.get("lanes", 1))
            self.scenes = [fg.Scene(self.ctx, p) for _, p, _ in self.members]

    def __del__(self):
        if self.server is not None:
            self.server.close()
        for s in self.scenes:
            s.close()
        self.ctx.close()

    def frames(self):
        for s, (_, _, objects) in zip(self.scenes, self.members):
            s.init_objects(**objects)
        for _ in range(self.case["frames"]):
            if self.case["kind"] == "hooks":
                self.frame_by_stages(self.scenes[0])
            elif len(self.scenes) > 1:
                fg.batch_step_frame(self.ctx, self.scenes)
            else:
                self.scenes[0].step_frame()
        return self.reader.read(self.scenes)

    def frame_by_stages(self, scene):
        """FlipSolver::stepFrame with step() as its stage hooks, as the C++ API runs an overriding subclass."""
        p, f = scene.params, np.float32
        frame_dt, t, count, last = f(1.0) / f(p.fps), f(0), 0, False
        while not last:
            dt = f(p.cfl_number) / (f(scene.max_velocity()) + f(1e-15))
            if t + dt >= frame_dt or count == p.max_substeps - 1:
                dt, last = frame_dt - t, True
            elif t + f(2) * dt >= frame_dt:
                dt = f(0.5) * (frame_dt - t)
            for stage in range(fg.STAGE_COUNT + 1):
                scene.stage(stage, float(dt))
            t, count = t + dt, count + 1

    def serve(self):
        ids = [self.server.submit(p, o["solids"], o["fluids"], m["frames"], seed=o["seed"], friction=o["friction"], keep=True)
               for m, p, o in self.members]
        while True:
            t = self.server.tick()
            if t.resident == 0 and t.queued == 0:
                break
        out = self.reader.read([self.server.scene(k) for k in ids])
        for k in ids:
            self.server.release(k)
        return out


# ---------------------------------------------------------------------------------------------------------------------
def prepare(case, seed):
    if case["kind"] == "solve":
        mat, b, scale = _system(case, seed)
        return {"ctx": fg.Context(0), "mat": mat.cpu().numpy(), "b": b.flatten().cpu().numpy(), "scale": scale,
                "noalloc": case["noalloc"]}
    return _Simulation(case, seed)


def run(state):
    if isinstance(state, dict):
        x, _ = state["ctx"].poisson_solve(state["mat"], state["scale"], state["b"], tol=TOL, noalloc=state["noalloc"])
        return {"pressure": x}
    return state.serve() if state.server is not None else state.frames()


def work(case):
    if case["kind"] == "solve":   # materials, right-hand side in, pressure out; one check of the result
        C = case["I"] * case["J"]
        return {"bytes": 17 * C, "flops": 10 * C}
    total = {"bytes": 0.0, "flops": 0.0}
    for m in [case] if case["kind"] in ("scene", "hooks") else _members(case):
        C = m["I"] * m["J"]
        x0, x1, y0, y1 = m.get("box", (0.3, 1.0, 0.0, 0.4)) if m["setup"] == "dam" else (0.6, 1.0, 0.0, 0.3)
        P = (x1 - x0) * (y1 - y0) * C * m["ppc"] * (0.1 if m["solver"] == "nbflip" else 1.0)
        # the first frame starts from rest (one substep); later ones need up to ten
        substeps = 1 + 8 * (m["frames"] - 1)
        # a substep reads and writes each particle (position, velocity, id), both velocity components, the materials
        # and the pressure, reads the solid and writes the fluid level set
        total["bytes"] += substeps * (40 * P + 16 * C + 2 * C + 16 * C + 8 * C) + 20 * P + 19 * C
        total["flops"] += substeps * (500 * P + 100 * C)
    return total
