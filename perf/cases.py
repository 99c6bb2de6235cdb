"""Measured cases of the smoke step: what a program that uses this framework has
it do, through the Python binding's public calls (smokesim.Simulation, Batch,
proxy_geometry).

A case is one of three kinds:
  * "sim"   -- one simulation advanced `steps` steps of dt = 0.05, then read
               (`reads`): "every" brings the density to the host after every
               step, as the reference's simulate() does; "last" reads it after
               the last step; "half" the same as a 16-bit read-back; "state"
               reads density, velocity, pressure and the step norms.
  * "batch" -- a batch of simulations of different sizes advanced `steps`
               steps (HIP-graph replay), then every member's density.
  * "proxy" -- one frame of the renderer's slicing geometry, host arrays.

Inputs: density blobs, a few large vortices of some cells per second plus
noise, seeded solid boxes and smoke sources, the benchmark scenes' physics.
exact() restates the step in FP64 with plain torch / numpy.
"""
import math
import os
import random
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                                "smoke-simulation_amd"))
import smokesim  # noqa: E402

DT = float(np.float32(0.05))
PHYSICS = dict(gravity=7.8, buoyancy=2.0, density_gate=0.001, max_velocity=4.0)
PROJECTION = {"reference": smokesim.PROJ_REFERENCE, "rbsor": smokesim.PROJ_RBSOR,
              "jacobi": smokesim.PROJ_JACOBI, "refined": smokesim.PROJ_REFINED}
STORAGE = {"fp32": smokesim.STORAGE_FP32, "bf16": smokesim.STORAGE_BF16,
           "fp16": smokesim.STORAGE_FP16, "fp16_velocity": smokesim.STORAGE_FP16_VELOCITY}

# Options of a "sim" case that are not given.
OPTIONS = dict(storage="fp32", iterations=60, inner_sweeps=20, steps=5, reads="last", boxes=0.05,
               sources=3, obstacles=0, moving=False, warm=False, vorticity=0.0, tuned=False,
               graph=False, norms=False)


def sim(name, dims, projection, **options):
    case = dict(kind="sim", nx=dims[0], ny=dims[1], nz=dims[2], projection=projection)
    case.update(OPTIONS)
    case.update(options)
    if name:
        case["name"] = name
    return case


def listed():
    return [
        # The renderer's frame: 100 slicing planes of the app's 80^3 box.
        dict(name="proxy_100", kind="proxy", planes=100, box=80.0),
        # The reference app's loop: its 80^3 volume, obstacle and source,
        # its own projection, the density back on the host every step.
        sim("app_80", (80, 80, 80), "reference", iterations=40, steps=1, reads="every", boxes=0.0,
            sources=1, obstacles=1),
        # The same loop in a larger ragged volume with the reference's default
        # 30 iterations and an obstacle the user drags (a new mask each step).
        sim("app_moving", (150, 96, 121), "reference", iterations=30, steps=4, reads="every",
            obstacles=2, moving=True),
        # The drop-in's projection at the larger benchmark grid's scale.
        sim("reference_256", (256, 240, 248), "reference", iterations=40, steps=2),
        # A small volume of a request's size, steps replayed from a graph.
        sim("small_48", (48, 40, 57), "jacobi", iterations=60, steps=10, graph=True),
        # Pressure-form SOR started from the last step's pressure, vorticity
        # confinement and per-step norms; the whole state is read.
        sim("warm_rbsor", (113, 90, 101), "rbsor", iterations=40, steps=5, reads="state", warm=True,
            vorticity=0.3, norms=True),
        # A ragged volume as a program that never tunes its plan runs it.
        sim("ragged_197", (197, 131, 243), "jacobi", iterations=60, steps=5),
        # 16-bit fields with the FP32 Jacobi solve, read back in 16 bits.
        sim("fp16_fields", (200, 169, 224), "jacobi", iterations=60, steps=5, reads="half",
            storage="fp16"),
        # The benchmark's 256^3 scene, plan tuned once by the program.
        sim("grid_256", (256, 256, 256), "jacobi", iterations=100, steps=10, sources=4, tuned=True),
        # 64 uneven volumes in one batch.
        dict(name="batch_64", kind="batch", count=64, lo=32, hi=160, iterations=60, steps=10,
             layout=64, tuned=True),
        # The headline: 512^3, 100 Jacobi sweeps.
        sim("grid_512", (512, 512, 512), "jacobi", iterations=100, steps=10, sources=8, tuned=True),
        # Its mixed-precision form: FP16 fields, 2 x 50 FP16 sweeps.
        sim("mixed_512", (512, 512, 512), "refined", iterations=100, inner_sweeps=50, steps=10,
            sources=8, storage="fp16", reads="half", tuned=True),
    ]


def log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["proxy", "batch", "sim", "sim", "sim", "sim", "sim", "sim"])
    if kind == "proxy":
        return dict(kind="proxy", planes=log_int(rng, 20, 4096), box=float(rng.randint(32, 512)))
    if kind == "batch":
        lo = rng.randint(16, 48)
        return dict(kind="batch", count=log_int(rng, 2, 64), lo=lo, hi=rng.randint(lo + 20, 160),
                    iterations=rng.choice([20, 30, 60]), steps=rng.randint(2, 10),
                    layout=rng.randint(1, 1 << 20), tuned=rng.random() < 0.5)
    side = math.exp(rng.uniform(math.log(20), math.log(320)))
    dims = tuple(max(12, min(400, int(round(side * rng.uniform(0.7, 1.4))))) for _ in range(3))
    projection = rng.choice(["reference", "reference", "rbsor", "jacobi", "jacobi", "refined"])
    options = dict(iterations=rng.choice([20, 30, 40, 60, 100]), steps=rng.randint(1, 8),
                   reads=rng.choice(["every", "last", "last", "state"]),
                   sources=rng.randint(1, 6), obstacles=rng.randint(0, 2),
                   boxes=rng.choice([0.0, 0.05, 0.1]))
    if projection == "reference":
        options["moving"] = options["obstacles"] > 0 and rng.random() < 0.5
    else:
        options["storage"] = rng.choice(["fp32", "fp32", "fp16", "bf16", "fp16_velocity"])
        options["tuned"] = projection != "rbsor" and rng.random() < 0.5
    if projection in ("rbsor", "jacobi"):
        options["warm"] = rng.random() < 0.4
    if projection == "refined":
        options.update(storage=rng.choice(["fp16", "fp16_velocity"]), inner_sweeps=20)
    if options.get("storage", "fp32") in ("fp16", "bf16") or projection == "refined":
        options["reads"] = "half"
    options["graph"] = rng.random() < 0.3
    options["norms"] = options["reads"] == "state"
    options["vorticity"] = rng.choice([0.0, 0.0, 0.3])
    return sim(None, dims, projection, **options)


# ------------------------------------------------------------------ inputs

def place_boxes(dims, fraction, rng):
    """The y = 0 floor plus axis-aligned boxes of edge 4..32 up to `fraction`
    of the cells (shape (nz, ny, nx), nonzero = solid)."""
    nx, ny, nz = dims
    solid = np.zeros((nz, ny, nx), np.uint8)
    solid[:, 0, :] = 1
    count, target = nx * nz, int(fraction * solid.size)
    while count < target:
        e = [min(rng.randint(4, 32), max(1, n // 3)) for n in dims]
        x, y, z = (rng.randint(0, n - k) for n, k in zip(dims, e))
        box = solid[z:z + e[2], y:y + e[1], x:x + e[0]]
        count += box.size - int(box.sum())
        box[...] = 1
    return solid


def place_spheres(dims, count, rng, top, radius):
    small = min(dims)
    out = []
    for _ in range(count):
        r = min(rng.uniform(*radius), small / 5.0)
        pos = (rng.uniform(r, dims[0] - r), rng.uniform(1.0, dims[1] * top),
               rng.uniform(r, dims[2] - r))
        out.append(tuple(float(np.float32(v)) for v in pos + (r,)))
    return out


def make_fields(dims, seed):
    """Initial density (nz, ny, nx) in [0, 1] and u, v, w (nz+1, ny+1, nx+1),
    made on the GPU, as host arrays."""
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    rng = random.Random(seed * 7 + 1)
    gen = torch.Generator(device=dev)
    gen.manual_seed(seed)
    nx, ny, nz = dims

    def wave(n, axis):
        c = torch.arange(n, device=dev, dtype=torch.float32)
        shape = [1, 1, 1]
        shape[axis] = n
        s = torch.sin(c * (2.0 * math.pi * rng.randint(1, 4) / n) + rng.uniform(0.0, 6.28))
        return s.reshape(shape)

    density = wave(nz, 0) * wave(ny, 1) * wave(nx, 2)
    density = torch.clamp(density * 1.2, 0.0, 1.0)
    velocity = []
    for k in range(3):
        a = torch.rand((nz + 1, ny + 1, nx + 1), device=dev, generator=gen)
        a = (a - 0.5) * 0.02
        for _ in range(2):
            a += wave(nz + 1, 0) * wave(ny + 1, 1) * wave(nx + 1, 2) * rng.uniform(0.5, 3.0)
        velocity.append(a.cpu().numpy())
    return density.cpu().numpy(), velocity


def make_scene(case, seed):
    rng = random.Random(seed)
    dims = (case["nx"], case["ny"], case["nz"])
    sc = dict(dims=dims)
    sc["solid"] = place_boxes(dims, case["boxes"], rng) if case["boxes"] else None
    sc["sources"] = place_spheres(dims, case["sources"], rng, 1.0 / 3.0, (3.0, 10.0))
    sc["obstacles"] = place_spheres(dims, case["obstacles"], rng, 1.0, (4.0, 14.0))
    sc["density"], sc["velocity"] = make_fields(dims, seed)
    return sc


def drag(scene, step):
    """Where the user has dragged the last obstacle before step `step`."""
    x, y, z, _ = scene["obstacles"][-1]
    return tuple(float(np.float32(p + 4.0 * math.sin(0.3 * step + k)))
                 for k, p in enumerate((x, y, z)))


def members(case):
    """The batch's member cases: the layout fixes their sizes."""
    rng = random.Random(case["layout"])
    out = []
    for _ in range(case["count"]):
        dims = tuple(rng.randint(case["lo"], case["hi"]) for _ in range(3))
        out.append(sim(None, dims, "jacobi", iterations=case["iterations"], steps=case["steps"],
                       boxes=rng.choice([0.0, 0.05, 0.1]), sources=rng.randint(1, 3)))
    return out


# The program's tuned plans: one per kind of grid, found by the autotuner the
# first time and set for every later simulation of that kind.
PLANS = {}


def tune(case, target):
    key = tuple(sorted((k, v) for k, v in case.items() if k not in ("name", "steps", "reads")))
    if key not in PLANS:
        PLANS[key] = target.autotune()[0]
    target.set_jacobi_plan(**PLANS[key])


def make_simulation(case, seed):
    scene = make_scene(case, seed)
    s = smokesim.Simulation(*scene["dims"], density=scene["density"],
                            storage=STORAGE[case["storage"]])
    if scene["solid"] is not None:
        s.set_solids(scene["solid"])
    ids = [s.add_obstacle(*o) for o in scene["obstacles"]]
    for o in scene["sources"]:
        s.add_source(*o)
    for k in range(3):
        s.set_velocity(k, 0, scene["velocity"][k])
    s.set_params(projection=PROJECTION[case["projection"]], iterations=case["iterations"],
                 inner_sweeps=case["inner_sweeps"], warm_start=1 if case["warm"] else 0,
                 vorticity=case["vorticity"], obstacle_mode=smokesim.OBSTACLES_UNION, **PHYSICS)
    if case["norms"]:
        s.norms_enable(True)
    if case["graph"]:
        s.set_step_graph(True)
    return s, scene, ids


def proxy_view(case, seed):
    rng = random.Random(seed)
    b = case["box"]
    direction = [rng.choice([-1.0, 1.0]) * rng.uniform(0.2, 1.0) for _ in range(3)]
    return ((0.0, 0.0, 0.0), (b, b * rng.uniform(0.5, 1.0), b * rng.uniform(0.5, 1.0)),
            (0.0, 0.0, 0.0), tuple(direction))


def prepare(case, seed):
    if case["kind"] == "proxy":
        return dict(case=case, view=proxy_view(case, seed))
    if case["kind"] == "batch":
        sims = [make_simulation(m, seed * 1000 + i)[0] for i, m in enumerate(members(case))]
        batch = smokesim.Batch(sims, [DT] * len(sims))
        if case["tuned"]:
            tune(case, batch)
        return dict(case=case, sims=sims, batch=batch)
    s, scene, ids = make_simulation(case, seed)
    if case["tuned"]:
        tune(case, s)
    return dict(case=case, sim=s, scene=scene, ids=ids, step=0)


def run(state):
    case = state["case"]
    if case["kind"] == "proxy":
        return smokesim.proxy_geometry(*state["view"], case["planes"])
    if case["kind"] == "batch":
        for _ in range(case["steps"]):
            state["batch"].step(use_graph=True)
        return [s.read_density() for s in state["sims"]]
    s = state["sim"]
    frames = []
    for _ in range(case["steps"]):
        state["step"] += 1
        if case["moving"]:
            s.move_object(state["ids"][-1], *drag(state["scene"], state["step"]))
        if case["reads"] == "every":
            frames.append(s.step(DT))
        else:
            s.step_async(DT)
    if case["reads"] == "every":
        return frames
    if case["reads"] == "half":
        s.readback_begin(smokesim.READBACK_F16)
        return s.readback_wait()[0]
    if case["reads"] == "last":
        return s.read_density()
    half = 1 - s.index_now
    out = dict(density=s.get_density(half), u=s.get_velocity(0, half), v=s.get_velocity(1, half),
               w=s.get_velocity(2, half), pressure=s.get_pressure())
    if case["norms"]:
        out["norms"] = s.step_norms()
    return out


# ------------------------------------------------------------------- work

def sim_work(case):
    """Each step reads and writes density and velocity once (the stored
    width) and reads the cell flags once; each relaxation of a cell is seven
    operations, the other stages about 250."""
    cells = case["nx"] * case["ny"] * case["nz"]
    width = {"fp32": 16, "fp16": 8, "bf16": 8, "fp16_velocity": 10}[case["storage"]]
    sweeps = case["iterations"]
    if case["projection"] == "refined":
        sweeps = math.ceil(sweeps / case["inner_sweeps"]) * case["inner_sweeps"]
    frames = case["steps"] if case["reads"] == "every" else 1
    read = {"half": 2, "state": 20}.get(case["reads"], 4) * frames
    return (cells * (case["steps"] * (2 * width + 1) + read),
            cells * case["steps"] * (7 * sweeps + 250))


def work(case):
    if case["kind"] == "proxy":
        return dict(bytes=case["planes"] * (7 * 12 + 18 * 2 + 8), flops=case["planes"] * 700)
    parts = [sim_work(c) for c in (members(case) if case["kind"] == "batch" else [case])]
    return dict(bytes=sum(p[0] for p in parts), flops=sum(p[1] for p in parts))


# --------------------------------------------------- the step in 64 bits

def cut(dims, x0=0, x1=0, y0=0, y1=0, z0=0, z1=0):
    """Slices [lo, n - 1 + hi] of a field of shape (nz+1, ny+1, nx+1)."""
    nx, ny, nz = dims
    return (slice(z0, nz + z1), slice(y0, ny + y1), slice(x0, nx + x1))


def move(a, dx=0, dy=0, dz=0):
    """The field whose value at (x, y, z) is a's at (x+dx, y+dy, z+dz) (what
    comes round from the other side is never used)."""
    return torch.roll(a, (-dz, -dy, -dx), (0, 1, 2))


class Exact:
    def __init__(self, case, seed):
        self.case = case
        self.scene = make_scene(case, seed)
        self.dims = nx, ny, nz = self.scene["dims"]
        self.dev = "cuda" if torch.cuda.is_available() else "cpu"
        shape = (nz + 1, ny + 1, nx + 1)
        new = lambda: torch.zeros(shape, dtype=torch.float64, device=self.dev)  # noqa: E731
        self.rho, self.vel = [new(), new()], [[new(), new()] for _ in range(3)]
        self.rho[0][:nz, :ny, :nx] = torch.from_numpy(self.scene["density"]).to(self.rho[0])
        for k in range(3):
            self.vel[k][0][...] = torch.from_numpy(self.scene["velocity"][k]).to(self.rho[0])
        self.pressure = new()
        self.now = 1
        solid = self.scene["solid"]
        if solid is None:
            solid = np.zeros((nz, ny, nx), np.uint8)
            solid[:, 0, :] = 1
        self.base = torch.zeros(shape, dtype=torch.bool, device=self.dev)
        self.base[:nz, :ny, :nx] = torch.from_numpy(solid).to(self.dev) == 0
        self.x, self.y, self.z = (torch.arange(n + 1, device=self.dev).reshape(s) for n, s in
                                  ((nx, (1, 1, -1)), (ny, (1, -1, 1)), (nz, (-1, 1, 1))))
        self.inner = ((self.x >= 1) & (self.x <= nx - 2) & (self.y >= 1) & (self.y <= ny - 2) &
                      (self.z >= 1) & (self.z <= nz - 2))
        p = dict(PHYSICS)
        self.prm = {k: float(np.float32(v)) for k, v in p.items()}
        self.mask(self.scene["obstacles"])

    def ball(self, sphere):
        """Cells inside a sphere, tested in FP32 as the scene defines it."""
        x, y, z, r = (torch.tensor(v, dtype=torch.float32) for v in sphere)
        d = [(c.to(torch.float32) - v.to(self.dev)) for c, v in
             ((self.x, x), (self.y, y), (self.z, z))]
        return ((d[0] * d[0] + d[1] * d[1] + d[2] * d[2]) < float(r * r)) & self.inner

    def mask(self, obstacles):
        s = self.base.clone()
        for o in obstacles:
            s &= ~self.ball(o)
        self.s = s
        # A neighbour counts only inside the grid: the padded cells are not fluid.
        nx, ny, nz = self.dims
        self.sm = [s & move(s, **{"d" + a: -1}) for a in "xyz"]
        for k, c in enumerate((self.x, self.y, self.z)):
            self.sm[k] &= c >= 1
        nb = [move(s, **{"d" + a: d}) for a in "xyz" for d in (-1, 1)]
        count = sum(n.to(torch.float64) for n in nb)
        self.active = self.inner & s & (count > 0)
        self.inv = torch.where(self.active, 1.0 / count.clamp(min=1.0), torch.zeros_like(count))
        self.nb = [n.to(torch.float64) for n in nb]

    def divergence(self):
        u, v, w = (self.vel[k][self.now] for k in range(3))
        d = move(u, dx=1) - u + move(v, dy=1) - v + move(w, dz=1) - w
        return torch.where(self.active, d, torch.zeros_like(d))

    def vorticity(self, eps):
        u, v, w = (self.vel[k][self.now] for k in range(3))
        cu, cv, cw = (u + move(u, dx=1)) / 2, (v + move(v, dy=1)) / 2, (w + move(w, dz=1)) / 2

        def der(a, axis):
            return (move(a, **{"d" + axis: 1}) - move(a, **{"d" + axis: -1})) / 2

        omega = [der(cw, "y") - der(cv, "z"), der(cu, "z") - der(cw, "x"),
                 der(cv, "x") - der(cu, "y")]
        here = self.inner & self.s
        omega = [torch.where(here, o, torch.zeros_like(o)) for o in omega]
        mag = torch.sqrt(omega[0] ** 2 + omega[1] ** 2 + omega[2] ** 2)
        e = [der(mag, a) for a in "xyz"]
        size = torch.sqrt(e[0] ** 2 + e[1] ** 2 + e[2] ** 2)
        ok = here & (size > 1e-6)
        n = [torch.where(ok, a / size, torch.zeros_like(a)) for a in e]
        for k, a in enumerate("xyz"):
            i, j = (k + 1) % 3, (k + 2) % 3
            f = eps * (n[i] * omega[j] - n[j] * omega[i])
            gain = DT * (f + move(f, **{"d" + a: -1})) / 2
            self.vel[k][self.now] += torch.where(self.sm[k], gain, torch.zeros_like(gain))

    def project(self):
        case, dims = self.case, self.dims
        parity = (self.x + self.y + self.z) % 2
        if case["projection"] == "reference":
            u, v, w = (self.vel[k][self.now] for k in range(3))
            for _ in range(case["iterations"]):
                for colour in range(2):
                    p = -self.divergence() * self.inv * 1.9 * (parity == colour)
                    for a, k in ((u, 0), (v, 1), (w, 2)):
                        a -= p * self.nb[2 * k]
                        a += move(p * self.nb[2 * k + 1], **{"d" + "xyz"[k]: -1})
            return
        d = self.divergence()
        p = self.pressure
        if case["warm"]:
            p *= self.active
        else:
            p.zero_()
        c = cut(dims, 1, -1, 1, -1, 1, -1)
        six = [cut(dims, 0, -2, 1, -1, 1, -1), cut(dims, 2, 0, 1, -1, 1, -1),
               cut(dims, 1, -1, 0, -2, 1, -1), cut(dims, 1, -1, 2, 0, 1, -1),
               cut(dims, 1, -1, 1, -1, 0, -2), cut(dims, 1, -1, 1, -1, 2, 0)]
        dc, inv = d[c], self.inv[c]
        g = torch.empty_like(dc)

        def relaxed(p):
            torch.add(p[six[0]], p[six[1]], out=g)
            for k in range(2, 6):
                g.add_(p[six[k]])
            return g.sub_(dc).mul_(inv)

        if case["projection"] == "rbsor":
            colours = [((parity[c] == k) & self.active[c]) * float(np.float32(1.9)) for k in (0, 1)]
            for _ in range(case["iterations"]):
                for k in range(2):
                    p[c] += (relaxed(p) - p[c]) * colours[k]
        else:
            sweeps = case["iterations"]
            if case["projection"] == "refined":
                sweeps = math.ceil(sweeps / case["inner_sweeps"]) * case["inner_sweeps"]
            for _ in range(sweeps):
                p[c] = relaxed(p)
        nx, ny, nz = dims
        low = ((self.x >= 1) & (self.x <= nx - 1) & (self.y >= 1) & (self.y <= ny - 1) &
               (self.z >= 1) & (self.z <= nz - 1))
        for k, a in enumerate("xyz"):
            diff = p - move(p, **{"d" + a: -1})
            self.vel[k][self.now] -= torch.where(self.sm[k] & low, diff, torch.zeros_like(diff))

    def sample(self, field, pos, shift):
        """The field at `pos`, its samples `shift` of a cell into each cell."""
        n = self.dims
        low, part = [], []
        for k in range(3):
            q = pos[k].clamp(1.0, n[k] - 1.0) - shift[k]
            i = torch.floor(q).clamp(max=n[k] - 1.0)
            part.append(q - i)
            low.append(i.long())
        high = [(low[k] + 1).clamp(max=n[k] - 1) for k in range(3)]
        row, plane = n[0] + 1, (n[0] + 1) * (n[1] + 1)
        flat, out = field.reshape(-1), 0.0
        for corner in range(8):
            at, weight = 0, 1.0
            for k, stride in ((0, 1), (1, row), (2, plane)):
                up = (corner >> k) & 1
                at = at + (high if up else low)[k] * stride
                weight = weight * (part[k] if up else 1.0 - part[k])
            out = out + flat[at] * weight
        return out

    def advect(self):
        nx, ny, nz = self.dims
        now, past = self.now, 1 - self.now
        u, v, w = (self.vel[k][now] for k in range(3))
        c = cut(self.dims, 1, 0, 1, 0, 1, 0)
        x, y, z = (torch.arange(1, n, device=self.dev, dtype=torch.float64).reshape(s) for n, s in
                   ((nx, (1, 1, -1)), (ny, (1, -1, 1)), (nz, (-1, 1, 1))))

        def mean(a, xs, ys, zs):
            return (sum(move(a, i, j, k) for i in xs for j in ys for k in zs) / 8.0)[c]

        back = (-1, 0)
        mu, mv, mw = mean(u, (0, 1), back, back), mean(v, back, (0, 1), back), mean(w, back, back, back)
        xm, ym, zm = x + 0.5 - DT * mu, y + 0.5 - DT * mv, z + 0.5 - DT * mw
        edge = [self.x[..., 1:nx] < nx - 1, self.y[:, 1:ny] < ny - 1, self.z[1:nz] < nz - 1]
        new = [self.sample(u, (x - DT * u[c], ym, zm), (0.0, 0.5, 0.5)),
               self.sample(v, (xm, y - DT * v[c], zm), (0.5, 0.0, 0.5)),
               self.sample(w, (xm, ym, z - DT * w[c]), (0.5, 0.5, 0.0))]
        for k in range(3):
            ok = self.sm[k][c] & edge[(k + 1) % 3] & edge[(k + 2) % 3]
            self.vel[k][past][c] = torch.where(ok, new[k], self.vel[k][past][c])
        del new, mu, mv, mw, xm, ym, zm
        c = cut(self.dims, 1, -1, 1, -1, 1, -1)
        u, v, w = (self.vel[k][past] for k in range(3))
        x, y, z = x[..., :-1], y[:, :-1], z[:-1]
        mid = [((a + move(a, **{"d" + b: 1})) / 2.0)[c] for a, b in ((u, "x"), (v, "y"), (w, "z"))]
        pos = (x + 0.5 - DT * mid[0], y + 0.5 - DT * mid[1], z + 0.5 - DT * mid[2])
        new = self.sample(self.rho[now], pos, (0.5, 0.5, 0.5))
        self.rho[past][c] = torch.where(self.s[c], new, self.rho[past][c])

    def step(self, obstacles=None):
        nx, ny, nz = self.dims
        if obstacles is not None:
            self.mask(obstacles)
        self.now = 1 - self.now
        for o in self.scene["sources"]:
            b = self.ball(o)
            self.rho[0][b] = 1.0
            self.rho[1][b] = 1.0
        prm, rho = self.prm, self.rho[self.now]
        u, v, w = (self.vel[k][self.now] for k in range(3))
        lift = (prm["gravity"] + prm["buoyancy"]) * DT * rho
        where = self.sm[1] & (rho > prm["density_gate"])
        v += torch.where(where, lift, torch.zeros_like(lift))
        box = ((self.x >= 1) & (self.x <= nx - 1) & (self.y >= 1) & (self.y <= ny - 1) &
               (self.z >= 1) & (self.z <= nz - 1))
        speed = (u * u + v * v + w * w) * DT
        most = prm["max_velocity"] ** 2
        scale = torch.where(box & (speed > most), most / speed, torch.ones_like(speed))
        for a in (u, v, w):
            a *= scale
        if self.case["vorticity"]:
            self.vorticity(float(np.float32(self.case["vorticity"])))
        self.project()
        self.advect()

    def density(self):
        nx, ny, nz = self.dims
        return self.rho[1 - self.now][:nz, :ny, :nx].clone()


def exact_sim(case, seed):
    e = Exact(case, seed)
    frames = []
    for k in range(case["steps"]):
        obstacles = None
        if case["moving"]:
            obstacles = list(e.scene["obstacles"])
            obstacles[-1] = drag(e.scene, k + 1) + obstacles[-1][3:]
        e.step(obstacles)
        if case["reads"] == "every":
            frames.append(e.density())
    if case["reads"] == "every":
        return frames
    if case["reads"] != "state":
        return e.density()
    nx, ny, nz = e.dims
    out = {name: e.vel[k][1 - e.now] for k, name in enumerate("uvw")}
    out["density"] = e.density()
    # The reference form leaves no pressure.
    out["pressure"] = (None if case["projection"] == "reference"
                       else e.pressure[:nz, :ny, :nx].clone())
    if case["norms"]:
        out["norms"] = None
    return out


def exact(case, seed):
    if case["kind"] == "proxy":
        # The first corner's opposite in a parallelogram lies on the sort key's
        # jump: which side it falls, and so the corners' order, is FP32 rounding.
        return None
    if case["kind"] == "batch":
        return [exact_sim(m, seed * 1000 + i) for i, m in enumerate(members(case))]
    return exact_sim(case, seed)
