"""The work that users of this package have it do, as cases to be timed.

Each case is one call sequence of a user's program through the package's
public entry points, on a tank of fluid whose particles and velocities are
made from a seed:

  step      `Simulation.sph_step()` of a DFSPH dam break: 2D and 3D, FP32 and
            FP64, with and without surface tension, 8 thousand to 4 million
            fluid particles
  mixture   the same call for a two-phase VFSPH mixture with drift and
            diffusion (FBM), surface tension and one viscosity per phase
  batch     `SceneBatch.step()`: many small independent dam breaks advanced
            together
  rollout   `adjoint.rollout()` and its backward pass: gradients with respect
            to the initial velocities, the viscosity and the surface tension
  surface   `Simulation.sph_step_reference()`: the step issued kernel by
            kernel through the sph.py names, as a program written for the
            reference's main loop issues it

One pass loads the state it starts from and takes one step (a rollout: a few
steps), so that every pass does the same work.  The particles start in the
cell order of a moment before, as they stand in a running simulation, where a
step moves few of them to another cell.  `exact` restates the step in 64 bits
with plain torch: neighbour pairs as index lists, sums by index_add, gradients
by autograd through them.
"""
import math

import numpy as np
import torch

from tichi_sph_amd import Config, Simulation
from tichi_sph_amd.adjoint import DiffRunner, rollout
from tichi_sph_amd.batch import SceneBatch

# Particle spacing (m) and speed of sound per kind of scene: those of the
# package's own scenario files.  dt = spacing / speed of sound.
SPACING = {2: 0.02, 3: 0.01}
SOUND = {2: 50, 3: 100}
MIX_SPACING, MIX_SOUND = 0.008, 80
WALL_LAYERS = {2: 3, 3: 2}
TAPE_BUDGET = 32 << 30  # bytes of HBM a differentiable run may keep its tapes in


# ---------------------------------------------------------------------------
# The cases
# ---------------------------------------------------------------------------
def step_case(nx, ny, nz, precision=4, gamma=0.0):
    return {"kind": "step", "nx": nx, "ny": ny, "nz": nz, "precision": precision, "gamma": gamma}


def mixture_case(nx, ny, nz):
    return {"kind": "mixture", "nx": nx, "ny": ny, "nz": nz, "precision": 4, "gamma": 0.07}


def batch_case(scenes, least, most, layout):
    return {"kind": "batch", "scenes": scenes, "least": least, "most": most, "layout": layout, "precision": 4,
            "gamma": 0.0}


def rollout_case(nx, ny, nz, steps, every, gamma):
    return {"kind": "rollout", "nx": nx, "ny": ny, "nz": nz, "steps": steps, "every": every, "precision": 4,
            "gamma": gamma}


def surface_case(nx, ny, nz):
    return {"kind": "surface", "nx": nx, "ny": ny, "nz": nz, "precision": 4, "gamma": 0.0}


def listed():
    return [
        # the 2D dam break scene and the small 3D one: interactive runs, where
        # launches and the host's share of a step count
        dict(step_case(128, 64, 0), name="step_2d_8k"),
        dict(step_case(20, 20, 20), name="step_3d_8k"),
        # double precision, odd sizes: reference solutions of a mid-sized tank
        dict(step_case(41, 37, 43, precision=8), name="step_3d_65k_f64"),
        # an ordinary scene with surface tension
        dict(step_case(50, 80, 50, gamma=0.07), name="step_3d_200k_tension"),
        # the package's headline scene, and a production-sized ragged one
        dict(step_case(100, 100, 100), name="step_3d_1m"),
        dict(step_case(161, 157, 159), name="step_3d_4m"),
        # the two-phase mixture scenes
        dict(mixture_case(16, 16, 16), name="mixture_3d_4k"),
        dict(mixture_case(125, 125, 125), name="mixture_3d_2m"),
        # data generation: independent scenes of uneven sizes at once
        dict(batch_case(24, 8000, 60000, 1), name="batch_24"),
        # inverse problems: the differentiable scene over a few steps, and the
        # gradient through one step of a large one without surface tension
        dict(rollout_case(50, 80, 50, 4, 2, 0.07), name="rollout_200k_tension"),
        dict(rollout_case(100, 100, 100, 1, 1, 0.0), name="rollout_1m"),
        # a program written against the reference's own main loop
        dict(surface_case(46, 47, 46), name="surface_3d_100k"),
    ]


def _block(rng, dim, least, most):
    """A block of about exp(uniform(log least, log most)) particles with
    uneven edges."""
    n = math.exp(rng.uniform(math.log(least), math.log(most)))
    edge = n ** (1.0 / dim)
    a, b = rng.uniform(0.75, 1.3), rng.uniform(0.75, 1.3)
    if dim == 2:
        return max(8, int(edge * a)), max(8, int(edge / a)), 0
    return max(8, int(edge * a)), max(8, int(edge * b)), max(8, int(edge / (a * b)))


def draw(rng):
    kind = rng.choice(["step", "step", "step", "step", "mixture", "batch", "rollout", "surface"])
    if kind == "step":
        dim = rng.choice([2, 3, 3])
        if dim == 3 and rng.random() < 0.2:
            return step_case(*_block(rng, 3, 4e3, 3e5), precision=8)
        if dim == 3 and rng.random() < 0.3:
            return step_case(*_block(rng, 3, 4e3, 1.5e6), gamma=round(rng.uniform(0.02, 0.1), 3))
        return step_case(*_block(rng, dim, 4e3, 3.5e6 if dim == 3 else 1e6))
    if kind == "mixture":
        return mixture_case(*_block(rng, 3, 3e3, 1.5e6))
    if kind == "batch":
        most = int(math.exp(rng.uniform(math.log(8e3), math.log(1e5))))
        return batch_case(rng.randint(4, 28), most // 5, most, rng.randint(0, 10 ** 6))
    if kind == "rollout":
        steps = rng.choice([1, 1, 2, 3, 4])
        return rollout_case(*_block(rng, 3, 5e3, 5e5), steps, rng.randint(1, steps), rng.choice([0.0, 0.05, 0.07]))
    return surface_case(*_block(rng, 3, 4e3, 1.6e5))


def _batch_blocks(case):
    """The blocks of a batch's scenes: sizes log-uniform, uneven edges."""
    g = np.random.default_rng(case["layout"])
    out = []
    for _ in range(case["scenes"]):
        n = math.exp(g.uniform(math.log(case["least"]), math.log(case["most"])))
        a, b = g.uniform(0.7, 1.4, 2)
        edge = n ** (1.0 / 3.0)
        out.append((max(6, int(edge * a)), max(6, int(edge / (a * b))), max(6, int(edge * b))))
    return out


# ---------------------------------------------------------------------------
# Scenes: configuration, particles and velocities from a seed
# ---------------------------------------------------------------------------
class Scene:
    """A block of fluid in a walled tank, on one lattice with its walls,
    slightly displaced and moving."""

    def __init__(self, kind, block, gamma, seed, relax=1.0):
        self.dim = d = 3 if block[2] else 2
        self.block = block = block[:d]
        mix = kind == "mixture"
        self.gps = MIX_SPACING if mix else SPACING[d]
        self.cs = MIX_SOUND if mix else SOUND[d]
        self.solver = "VFSPH" if mix else "DFSPH"
        self.phases = 2 if mix else 1
        self.rho = [1000, 500][: self.phases]
        self.mu = 0.01
        self.phase_mu = [0.01, 0.05] if mix else None
        self.gamma = gamma
        self.fbm_d, self.fbm_c = (1e-4, 50) if mix else (0.0, 50)
        # A mixture's and a rollout's tank is closed and full, the others are
        # dam breaks.  `relax` is the scenarios' particle_relaxing_factor.
        self.closed = kind in ("mixture", "rollout")
        self.relax = relax
        self.threshold = 0.1 if kind == "rollout" else 1e-3
        self.jitter = 0.004
        s = self.gps * self.relax
        layers = WALL_LAYERS[d]
        inner = list(block)
        if not self.closed:
            inner[0] = 2 * block[0]
            inner[1] = block[1] + max(4, block[1] // 4)
        # the grid: two spacings of padding beyond the walls
        self.lb = [round(-(layers + 2) * s, 9)] * d
        self.rt = [round((n + layers + 2) * s, 9) for n in inner]
        g = np.random.default_rng([seed, 7, *block])
        axes = [np.arange(n) for n in block]
        idx = np.stack(np.meshgrid(*axes, indexing="ij"), axis=-1).reshape(-1, d)
        x = (idx + 0.49) * s
        x += g.uniform(-1, 1, x.shape) * (self.jitter * s)
        # smooth motion of a few decimetres per second, and some noise
        size = np.array(inner) * s
        v = g.normal(0, 0.005, x.shape)
        for _ in range(3):
            wave = g.uniform(0.5, 1.5, d) * math.pi / size
            phase = g.uniform(0, 2 * math.pi)
            v += np.sin(x @ wave + phase)[:, None] * g.normal(0, 0.1, d)
        self.top = idx[:, 1] >= block[1] // 2  # a mixture's second phase
        # cell order of a moment before (x fastest), ascending index in a cell
        dt = self.gps / self.cs
        order = np.argsort(self.keys((x - dt * v).astype(np.float32), np.float32), kind="stable")
        self.x, self.v, self.top = x[order].astype(np.float32), v[order].astype(np.float32), self.top[order]
        shape = [n + 2 * layers for n in inner]
        box = np.ones(shape, dtype=bool)
        box[tuple(slice(layers, n - layers) for n in shape)] = False
        self.xb = ((np.stack(np.where(box), axis=1) - layers + 0.49) * s).astype(np.float32)

    def keys(self, x, t):
        """Cell keys of positions, computed in type t: floor((x - lb) / h)."""
        h = t(np.float32(2 * np.float32(self.gps)))
        c = [np.floor((x[:, a].astype(t) - t(np.float32(self.lb[a]))) / h).astype(np.int64) for a in range(self.dim)]
        key, step = c[0].copy(), 1
        for a in range(1, self.dim):
            step *= self.grid()[a - 1]
            key += c[a] * step
        return key

    def grid(self):
        f = np.float32
        return [int(np.ceil((f(self.rt[a]) - f(self.lb[a])) / f(2 * f(self.gps)))) for a in range(self.dim)]

    def config(self):
        solver = {
            "arch": "gpu", "device_memory_GB": 6, "solver_type": self.solver, "solver_wc_gamma": 7,
            "solver_divergence_threshold": self.threshold, "solver_compression_threshold": self.threshold,
            "solver_iter_threshold_min": 2, "solver_iter_threshold_max": 100, "solver_if_cfl": True,
            "solver_cs": self.cs, "solver_cfl_factor": 0.5, "solver_neighb_range": 1,
            "solver_neighb_grid_size_TO_global_part_size": 2, "solver_fbm_diffusion_term": self.fbm_d,
            "solver_fbm_convection_term": self.fbm_c, "solver_surface_tension_gamma": self.gamma,
            "gui_res": [1080, 1080], "gui_part_zoomer": 1.0, "gui_fps": 30,
            "gui_canvas_bgcolor": [0.2, 0.2, 0.6], "gui_camera_pos": [6.0, 1.0, 0.0],
            "gui_camera_lookat": [0.0, 0.0, 0.0],
        }
        env = {
            "global_part_size": self.gps, "global_dynamic_viscosity": self.mu, "sim_dim": self.dim,
            "sim_space_lb": self.lb, "sim_space_rt": self.rt, "gravity": [0, -9.81, 0][: self.dim],
            "phase_num": self.phases, "phase_rest_density": self.rho,
            "phase_color_hex": ["0x6F7DBC", "0xFA8012"][: self.phases],
        }
        if self.phase_mu:
            env["phase_dynamic_viscosity"] = self.phase_mu
        return Config(solver, {"sim_env": env, "fluid": {"max_part_num": len(self.x), "objs": []},
                               "bound": {"max_part_num": len(self.xb), "objs": []}})

    def simulation(self, precision, **kw):
        """The Simulation of this scene, its fluid in the order of self.x."""
        sim = Simulation(self.config(), precision=precision, **kw)
        zero = [0.0] * self.dim
        one = [1] + [0] * (self.phases - 1)
        sim.fluid.push_part_seq(len(self.x), self.x, one, zero)
        sim.fluid.from_numpy("vel", self.v)
        if self.phases == 2:
            sim.fluid.from_numpy("volume_frac", np.stack([~self.top, self.top], axis=1).astype(np.float32))
            sim.fluid.update_mass_all()
        sim.bound.push_part_seq(len(self.xb), self.xb, one, zero)
        return sim


def _scene(case, seed):
    # A gradient is that of the recorded path, and the solves' clamp at zero
    # pressure breaks it: a particle whose clamp turns over by rounding alone
    # changes the gradient.  A rollout of one step starts from particles a
    # little closer than at rest (all under pressure, no clamp acts), a longer
    # one from a little wider (no pressure, every clamp holds), so that its
    # result can be compared; both leave the minimum number of iterations.
    relax = 1.0
    if case["kind"] == "rollout":
        relax = 0.995 if case["steps"] == 1 else 1.01
    return Scene(case["kind"], (case["nx"], case["ny"], case["nz"]), case["gamma"], seed, relax)


def _saved(sim, names):
    f = sim.fluid
    return {name: f.t[name][: f.part_num].clone() for name in names}


# ---------------------------------------------------------------------------
# What a program has in hand, and one pass
# ---------------------------------------------------------------------------
# The state a pass starts from.  The masses, densities and volumes of a
# one-phase fluid are the same for all its particles.
ONE_PHASE = ("pos", "vel", "pid")
MIXTURE = ("pos", "vel", "pid", "mass", "rest_density", "rest_volume", "volume_frac")


def prepare(case, seed):
    kind = case["kind"]
    if kind == "step":
        sim = _scene(case, seed).simulation(case["precision"])
        return {"kind": kind, "sim": sim, "start": _saved(sim, ONE_PHASE)}
    if kind == "mixture":
        sim = _scene(case, seed).simulation(case["precision"], fbm=True)
        return {"kind": kind, "sim": sim, "start": _saved(sim, MIXTURE)}
    if kind == "surface":
        sim = _scene(case, seed).simulation(case["precision"])
        return {"kind": kind, "sim": sim, "start": _saved(sim, ("pos", "vel"))}
    if kind == "batch":
        sims = []
        for k, block in enumerate(_batch_blocks(case)):
            scene = Scene(kind, block, case["gamma"], 1000 * seed + k)
            # particles in the order of this step: a batch's scenes differ in
            # which buffers hold their state, never in the order of it
            order = np.argsort(scene.keys(scene.x, np.float32), kind="stable")
            scene.x, scene.v = scene.x[order], scene.v[order]
            sims.append(scene.simulation(case["precision"], cfl=False))
        batch = SceneBatch(sims)
        start = [_saved(sim, ("pos", "vel")) for sim in sims]
        # the two buffers that the sort's swap alternates between
        live = [[sim.fluid.t[name + back][: sim.fluid.part_num] for sim in sims for name in ("pos", "vel")]
                for back in ("", "_b")]
        return {"kind": kind, "batch": batch, "live": live, "turn": 0,
                "start": [s[name] for s in start for name in ("pos", "vel")]}
    scene = _scene(case, seed)
    sim = scene.simulation(case["precision"], cfl=False)
    runner = DiffRunner(sim)
    g = np.random.default_rng([seed, 11])
    dev, dt = sim.device, sim.fluid.dtype
    target = torch.as_tensor(scene.x + g.normal(0, 0.002, scene.x.shape), dtype=dt, device=dev)
    return {"kind": kind, "runner": runner, "start": runner.checkpoint(), "target": target,
            "v0": torch.as_tensor(scene.v, dtype=dt, device=dev), "mu": scene.mu, "gamma": case["gamma"],
            "steps": case["steps"], "every": case["every"]}


def _load(sim, start):
    f = sim.fluid
    for name, t in start.items():
        f.t[name][: f.part_num].copy_(t)


def run(state):
    kind = state["kind"]
    if kind == "batch":
        batch = state["batch"]
        torch._foreach_copy_(state["live"][state["turn"]], state["start"])
        state["turn"] ^= 1
        batch.step()
        return [{"pos": s.fluid.t["pos"][: s.fluid.part_num], "vel": s.fluid.t["vel"][: s.fluid.part_num]}
                for s in batch.sims]
    if kind == "rollout":
        runner, v0 = state["runner"], state["v0"]
        runner.restore(state["start"])
        v = v0.clone().requires_grad_(True)
        mu = torch.tensor(state["mu"], dtype=v.dtype, device=v.device, requires_grad=True)
        gamma = torch.tensor(state["gamma"], dtype=v.dtype, device=v.device, requires_grad=state["gamma"] != 0)
        x, vel = rollout(runner, v, mu, gamma, state["steps"], state["every"], tape_budget=TAPE_BUDGET)
        (((x - state["target"]) ** 2).sum() + 1e-4 * (vel ** 2).sum()).backward()
        out = {"pos": x.detach(), "vel": vel.detach(), "grad_v": v.grad, "grad_mu": mu.grad}
        if state["gamma"] != 0:
            out["grad_gamma"] = gamma.grad
        return out
    sim = state["sim"]
    f, b = sim.fluid, sim.bound
    n = f.part_num
    _load(sim, state["start"])
    if kind == "surface":
        sim.sph_step_reference()
        return {"pos": f.t["pos"][:n], "vel": f.t["vel"][:n], "density": f.t["sph_density"][:n],
                "normal": f.t["normal"][:n], "wall_density": b.t["sph_density"][: b.part_num]}
    sim.sph_step()
    out = {"pos": f.t["pos"][:n], "vel": f.t["vel"][:n], "pid": f.t["pid"][:n], "density": f.t["sph_density"][:n],
           "alpha": f.t["alpha"][:n], "wall_density": b.t["sph_density"][: b.part_num]}
    if kind == "mixture":
        out["volume_frac"] = f.t["volume_frac"][:n]
        out["mass"] = f.t["mass"][:n]
    return out


def _particles(block):
    """(fluid, wall) particles of a block's tank, without making it."""
    return block[0] * block[1] * (block[2] or 1)


def work(case):
    """One step reads each particle's state (position, velocity, mass, rest
    density, rest volume, fractions, index) once and writes it once; its
    operations are those of the pair sums over about 30 (3D) or 14 (2D)
    neighbours within the support: density and alpha, two iterations of each
    solve, advection, and the reverse of each in a rollout."""
    s = case["precision"]
    blocks = _batch_blocks(case) if case["kind"] == "batch" else [(case["nx"], case["ny"], case["nz"])]
    d = 3 if blocks[0][2] else 2
    n = sum(_particles(b) for b in blocks)
    phases = 2 if case["kind"] == "mixture" else 1
    state = n * ((2 * d + 3 + phases) * s + 4)
    pairs = n * (30 if d == 3 else 14)
    sweep = pairs * (40 + 4 * (22 + 16) + 32 + (30 if case["gamma"] else 0) + (40 if phases == 2 else 0))
    if case["kind"] == "rollout":
        return {"bytes": 2 * state * 2, "flops": case["steps"] * (sweep + 2.5 * sweep)}
    return {"bytes": 2 * state, "flops": sweep}


# ---------------------------------------------------------------------------
# The step in 64 bits
# ---------------------------------------------------------------------------
def _f(x):
    """A constant as the scenario reader keeps it: rounded to 32 bits."""
    return float(np.float32(x))


class Exact:
    """The scene's step in 64 bits.  Which cell a particle is in is decided
    in the precision that the simulation runs in, as that choice is part of
    the step's definition."""

    def __init__(self, scene, precision):
        self.sc, self.precision = scene, precision
        d = self.d = scene.dim
        self.dev = torch.device("cuda" if torch.cuda.is_available() else "cpu")
        self.h = _f(2 * np.float32(scene.gps))
        self.h2 = _f(self.h ** 2)
        self.sig = _f(8 / math.pi / self.h ** 3) if d == 3 else _f(40 / 7 / math.pi / self.h ** 2)
        self.eps = 0.01 * self.h2
        self.vol = _f(_f(scene.gps) ** d)
        self.dt = _f(scene.gps) / scene.cs if precision == 8 else _f(np.float32(scene.gps) / np.float32(scene.cs))
        self.grav = self.t([0, _f(-9.81), 0][:d])
        self.rho = self.t([_f(r) for r in scene.rho])
        self.xb = self.t(scene.xb)
        n, nb = len(scene.x), len(scene.xb)
        phi = np.stack([~scene.top, scene.top], axis=1) if scene.phases == 2 else np.ones((n, 1))
        self.phi = self.t(phi)
        self.rest = (self.phi * self.rho).sum(1)
        self.mass = self.t((self.rest.cpu().numpy().astype(np.float32) * np.float32(self.vol)))
        self.massb = self.t(np.full(nb, np.float32(scene.rho[0]) * np.float32(self.vol)))
        self.vfsph = scene.solver == "VFSPH"
        self.X = torch.full_like(self.mass, self.vol) if self.vfsph else self.mass
        self.Xb = torch.full_like(self.massb, self.vol) if self.vfsph else self.massb
        mu = [_f(m) for m in scene.phase_mu] if scene.phase_mu else [_f(scene.mu)]
        self.mu = (self.phi * self.t(mu)).sum(1)
        self.gamma = _f(scene.gamma)

    def t(self, a):
        return torch.as_tensor(np.asarray(a, dtype=np.float64), device=self.dev)

    def keys(self, x):
        f = np.float32 if self.precision == 4 else np.float64
        return torch.as_tensor(self.sc.keys(x.detach().cpu().numpy().astype(f), f), device=self.dev)

    def candidates(self, xa, xb):
        """Yields (i, j) index pairs: j of xb in the cells around i of xa's,
        in chunks."""
        grid = self.sc.grid()
        ka, kb = self.keys(xa), self.keys(xb)
        order = torch.argsort(kb, stable=True)
        cells = 1
        for g in grid:
            cells *= g
        start = torch.zeros(cells + 1, dtype=torch.int64, device=self.dev)
        start[1:] = torch.cumsum(torch.bincount(kb, minlength=cells), 0)
        row, plane = grid[0], grid[0] * grid[1]
        i = torch.arange(len(xa), device=self.dev)
        for dz in ((-1, 0, 1) if self.d == 3 else (0,)):
            for dy in (-1, 0, 1):
                c = ka + dy * row + dz * plane
                lo, hi = start[c - 1], start[c + 2]
                for m in range(int((hi - lo).max())):
                    at = lo + m
                    ok = at < hi
                    yield i[ok], order[at[ok]]

    def pairs(self, xa, xb):
        """The pairs with 0 < r < h of xa's particles and xb's."""
        got = []
        for i, j in self.candidates(xa, xb):
            r2 = ((xa[i] - xb[j]) ** 2).sum(1)
            ok = (r2 > 0) & (r2 < self.h * self.h)
            got.append((i[ok], j[ok]))
        i, j = torch.cat([a for a, _ in got]), torch.cat([b for _, b in got])
        del got
        return i, j

    def geometry(self, xa, xb, ij):
        """x_ij, r, W, W'(r) / r of the pairs."""
        i, j = ij
        x = xa[i] - xb[j]
        r = (x * x).sum(1).sqrt()
        q = r / self.h
        near = q <= 0.5
        w = torch.where(near, 6 * (q ** 3 - q ** 2) + 1, 2 * (1 - q) ** 3) * self.sig
        g = torch.where(near, 6 * (3 * q - 2) / self.h ** 2, -6 * (1 - q) ** 2 / (self.h * r)) * self.sig
        return x, r, w, g

    @staticmethod
    def add(n, i, v):
        out = torch.zeros((n,) + v.shape[1:], dtype=v.dtype, device=v.device)
        return out.index_add(0, i, v)

    def density(self, x, ff, fb):
        n = len(x)
        xj, _, w, g = self.geometry(x, x, ff)
        xk, _, wb, gb = self.geometry(x, self.xb, fb)
        j, k = ff[1], fb[1]
        w0 = self.sig
        dens = w0 * self.mass + self.add(n, ff[0], w * self.mass[j]) + self.add(n, fb[0], wb * self.massb[k])
        comp = w0 * self.vol + self.add(n, ff[0], w * self.vol) + self.add(n, fb[0], wb * self.vol)
        a1 = self.add(n, ff[0], (self.X[j] * g)[:, None] * xj)
        a1 = a1 + self.add(n, fb[0], (self.Xb[k] * gb)[:, None] * xk)
        r2 = (xj * xj).sum(1)
        a2 = self.add(n, ff[0], g * g * r2 * self.X[j] ** 2 / self.mass[j])
        alpha = (a1 * a1).sum(1) / self.mass + a2
        return dens, comp, torch.clamp(alpha, min=1e-4)

    def iteration(self, x, va, psi0, rest, alpha, ff, fb):
        """One iteration of a solve: the new velocities and the error."""
        n = len(x)
        xj, _, _, g = self.geometry(x, x, ff)
        xk, _, _, gb = self.geometry(x, self.xb, fb)
        i, j = ff
        i2, k = fb
        s = self.add(n, i, ((va[i] - va[j]) * xj).sum(1) * g * self.X[j])
        s = s + self.add(n, i2, (va[i2] * xk).sum(1) * gb * self.Xb[k])
        psi = torch.clamp(psi0 - rest + self.dt * s, min=0)
        kap = psi / alpha
        up = self.add(n, i, ((kap[i] * self.X[j] + kap[j] * self.X[i]) * g)[:, None] * xj)
        up = up + self.add(n, i2, (kap[i2] * self.Xb[k] * gb)[:, None] * xk)
        return va - up / self.dt / self.mass[:, None], (psi / rest).mean()

    def solve(self, x, va, psi0, rest, alpha, ff, fb, ck):
        it = 0
        while True:
            va, err = ck(self.iteration, x, va, psi0, rest, alpha, ff, fb)
            it += 1
            if it >= 2 and (it > 100 or not float(err.detach()) > self.sc.threshold):
                return va

    def advection(self, x, v, psi, mu, gamma, ff):
        """gravity + viscosity + surface tension, without the curvature."""
        n = len(x)
        xj, r, _, g = self.geometry(x, x, ff)
        i, j = ff
        V = (self.X / psi)[j]
        lap = 2 * (2 + self.d) * V * g * ((v[i] - v[j]) * xj).sum(1) / (self.eps + r * r)
        acc = self.grav + self.add(n, i, lap[:, None] * xj) * (mu / self.rest)[:, None]
        normal = self.add(n, i, -(V * g)[:, None] * xj) * self.h
        if self.sc.gamma:
            q = r / self.h
            c = torch.where(q <= 0.5, 2 * (1 - q) ** 3 * q ** 3 - 1 / 64, (1 - q) ** 3 * q ** 3)
            c = c * (32 / math.pi / self.h ** 3) * self.gated[i] * self.gated[j]
            f = 2 * self.rest_psi()[i] / (psi[i] + psi[j])
            acc = acc - gamma * self.add(n, i, (f * self.mass[j] * c / r)[:, None] * xj)
        return acc, normal

    def rest_psi(self):
        return torch.ones_like(self.rest) if self.vfsph else self.rest

    def curvature(self, normal, psi, i, j):
        f = 2 * self.rest_psi()[i] / (psi[i] + psi[j]) * self.gated[i] * self.gated[j]
        return self.add(len(psi), i, f[:, None] * (normal[i] - normal[j]))

    def step(self, x, v, mu, gamma, ck=lambda f, *a: f(*a)):
        """The step from (x, v); mu and gamma may be differentiated."""
        with torch.no_grad():
            ff, fb = self.pairs(x, x), self.pairs(x, self.xb)
        self.gated = (self.phi[:, 0] > 0.99).to(torch.float64)
        dens, comp, alpha = ck(self.density, x, ff, fb)
        psi, rest = (comp if self.vfsph else dens), self.rest_psi()
        v = self.solve(x, v, psi, rest, alpha, ff, fb, ck)
        acc, normal = ck(self.advection, x, v, psi, mu, gamma, ff)
        if self.sc.gamma:  # over all candidates: it carries no kernel
            with torch.no_grad():
                lists = [(i[i != j], j[i != j]) for i, j in self.candidates(x, x)]
            for part in range(0, len(lists), 16):
                i = torch.cat([a for a, _ in lists[part:part + 16]])
                j = torch.cat([b for _, b in lists[part:part + 16]])
                acc = acc + gamma * ck(self.curvature, normal, psi, i, j)
            del lists
        va = self.solve(x, v + acc * self.dt, psi, rest, alpha, ff, fb, ck)
        if self.sc.phases == 2:
            self.mix(x, v, va, ff)
        self.dens, self.alpha, self.normal = dens, alpha, normal
        return x + va * self.dt, va

    def mix(self, x, v, va, ff):
        """The drift and diffusion of the volume fractions."""
        n, (i, j) = len(x), ff
        xj, r, _, g = self.geometry(x, x, ff)
        aa = (va - v) / self.dt
        z = (self.phi * (self.rho - self.rest[:, None]) / self.rho).sum(1)
        fa = (aa - z[:, None] * self.grav) / (1 - z)[:, None]
        flag = torch.zeros(n, dtype=torch.bool, device=self.dev)
        while True:
            tmp = torch.zeros_like(self.phi)
            live = (~flag[i] & ~flag[j]).to(torch.float64)
            for p in range(2):
                phi = self.phi[:, p]
                w = phi * self.rho[p]
                u = (phi * (self.rho[p] - self.rest))[:, None] * (self.grav - fa)
                u = torch.where((w > 1e-6)[:, None], u / torch.clamp(w, min=1e-30)[:, None], 0 * u)
                u = (u + (fa - aa)) * self.dt
                flux = phi[:, None] * u
                conv = self.add(n, i, live * ((flux[i] + flux[j]) * xj).sum(1) * g * self.vol)
                diff = self.add(n, i, live * (phi[i] - phi[j]) * self.vol * r * r * g / (r * r + self.eps))
                tmp[:, p] = -_f(self.sc.fbm_c) * self.dt * conv + self.dt * _f(self.sc.fbm_d) * diff
            tmp[flag] = 0
            new = ((self.phi + tmp) < 0).any(1)
            if not bool((new & ~flag).any()):
                break
            flag |= new
        self.phi = torch.where(flag[:, None], self.phi, self.phi + tmp)
        self.rest = (self.phi * self.rho).sum(1)
        self.mass = self.rest * self.vol

    def wall_density(self, x):
        nb = len(self.xb)
        bb, bf = self.pairs(self.xb, self.xb), self.pairs(self.xb, x)
        w = self.geometry(self.xb, self.xb, bb)[2]
        wf = self.geometry(self.xb, x, bf)[2]
        return (self.sig * self.massb + self.add(nb, bb[0], w * self.massb[bb[1]])
                + self.add(nb, bf[0], wf * self.mass[bf[1]]))


def _vec4(a, w=None):
    """[n, d] as the package keeps vectors: four lanes."""
    out = torch.zeros(len(a), 4, dtype=a.dtype, device=a.device)
    out[:, : a.shape[1]] = a
    if w is not None:
        out[:, 3] = w
    return out


def _exact_step(scene, precision, kind):
    e = Exact(scene, precision)
    x, v = e.t(scene.x), e.t(scene.v)
    wall = e.wall_density(x) if kind != "batch" else None
    x1, v1 = e.step(x, v, e.mu, e.gamma)
    w = e.X if e.vfsph else e.rest * e.vol
    if kind == "surface":
        return {"pos": _vec4(x1, w), "vel": _vec4(v1), "density": e.dens, "normal": _vec4(e.normal),
                "wall_density": wall}
    order = torch.argsort(e.keys(x), stable=True)  # the step keeps its particles in cell order
    out = {"pos": _vec4(x1, w)[order], "vel": _vec4(v1)[order]}
    if kind == "batch":
        return out
    at = torch.argsort(torch.as_tensor(scene.keys(scene.xb, np.float32 if precision == 4 else np.float64),
                                       device=e.dev), stable=True)
    out.update(pid=order.to(torch.int32), density=e.dens[order], alpha=e.alpha[order], wall_density=wall[at])
    if kind == "mixture":
        out.update(volume_frac=e.phi[order], mass=e.mass[order])
    return out


def exact(case, seed):
    kind = case["kind"]
    if kind == "batch":
        out = []
        for k, block in enumerate(_batch_blocks(case)):
            out.append(_exact_step(Scene(kind, block, case["gamma"], 1000 * seed + k), case["precision"], kind))
        return out
    scene = _scene(case, seed)
    if kind != "rollout":
        return _exact_step(scene, case["precision"], kind)
    if len(scene.x) * case["steps"] > 1e6:  # over 20 seconds, and more memory than the card has
        return None
    from torch.utils.checkpoint import checkpoint

    def ck(f, *a):
        return checkpoint(f, *a, use_reentrant=False)

    e = Exact(scene, case["precision"])
    g = np.random.default_rng([seed, 11])
    target = e.t((scene.x + g.normal(0, 0.002, scene.x.shape)).astype(np.float32))
    x, v0 = e.t(scene.x), e.t(scene.v).requires_grad_(True)
    mu = torch.full((), _f(scene.mu), dtype=torch.float64, device=e.dev, requires_grad=True)
    gamma = torch.full((), _f(scene.gamma), dtype=torch.float64, device=e.dev, requires_grad=True)
    v = v0
    for _ in range(case["steps"]):
        x, v = e.step(x, v, mu, gamma, ck)
    (((x - target) ** 2).sum() + 1e-4 * (v ** 2).sum()).backward()
    out = {"pos": x.detach(), "vel": v.detach(), "grad_v": v0.grad, "grad_mu": mu.grad}
    if case["gamma"] != 0:
        out["grad_gamma"] = gamma.grad
    return out
