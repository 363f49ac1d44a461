"""Performance cases of the framework: what its users have it do, from the smallest calls to the
largest, through the public entry points.

``listed()`` gives the fixed cases, ``draw(rng)`` one more of the same ranges.  ``prepare`` builds
what a program holds before the call (fields, masks, stepper), ``run`` is one pass, ``work`` the
bytes and operations a pass cannot do without, and ``exact`` the same outputs in float64 by plain
torch, from the definitions of the lattice-Boltzmann step and its boundary conditions.

Kinds of case (``"kind"``):

* ``loop``    -- the caller's own loop ``f_0, f_1 = stepper(...); f_0, f_1 = f_1, f_0``;
* ``run``     -- the same loop through ``stepper.run``;
* ``rollout`` -- a differentiable rollout, forward and backward;
* ``observe`` -- what a program looks at between steps: moments, vorticity and Q-criterion.

Geometries (``"flow"``): ``periodic`` (no boundary cells), ``cavity`` (a lid and five, or three,
bounce-back walls), ``channel`` (2-D: regularized inlet, extrapolation outlet, halfway walls and a
body-force field) and ``tunnel`` (3-D: regularized inlet, extrapolation outlet, full-way walls and a
halfway bounce-back sphere, with the drag at the end).
"""

import itertools
import math

import torch
from torch.utils.checkpoint import checkpoint

import xlb_amd as xa

# ------------------------------------------------------------------------------------------------
# The cases
# ------------------------------------------------------------------------------------------------
STORE = {"FP32FP32": torch.float32, "FP32FP32_DEVIATION": torch.float32, "FP64FP64": torch.float64,
         "FP32FP16_SHIFTED": torch.float16, "FP32I16_BLOCK": torch.int16}
LID = 0.02  # lid speed and the velocity scale of the initial flows
SMAGORINSKY = 0.17


def _case(name, kind, flow, lattice, shape, steps, policy="FP32FP32", collision="BGK", omega=1.0, walls="fullway"):
    nx, ny, nz = tuple(shape) + (1,) * (3 - len(shape))
    c = dict(kind=kind, flow=flow, lattice=lattice, nx=nx, ny=ny, nz=nz, steps=steps, policy=policy,
             collision=collision, omega=omega, walls=walls)
    if name:
        c["name"] = name
    return c


def listed():
    return [
        # a small 2-D cavity stepped from Python, as the 2-D example does: a few thousand cells per
        # call, so the cost of a call is what counts
        _case("loop_cavity2d_64", "loop", "cavity", "D2Q9", (64, 64), 20, omega=1.4, walls="halfway"),
        # a 3-D LES cavity of odd extents stepped from Python
        _case("loop_les_101x83x77", "loop", "cavity", "D3Q19", (101, 83, 77), 10, collision="SmagorinskyLESBGK",
              omega=1.9, walls="halfway"),
        # the 2-D forced channel of the differentiable workload, simulated only
        _case("run_channel2d_512x256", "run", "channel", "D2Q9", (512, 256), 100, omega=1.6),
        # the 64^3 lid-driven cavity: fields that fit the caches
        _case("run_cavity_64", "run", "cavity", "D3Q19", (64, 64, 64), 100, walls="halfway", omega=1.5),
        # the headline benchmark: the 256^3 lid-driven cavity in FP32
        _case("run_cavity_256", "run", "cavity", "D3Q19", (256, 256, 256), 40),
        # a Taylor-Green-sized periodic box, the largest field of the benchmark
        _case("run_periodic_512x256x256", "run", "periodic", "D3Q19", (512, 256, 256), 20, omega=1.9),
        # double precision, as used for validation, on a grid of no special size
        _case("run_periodic_fp64_150x90x110", "run", "periodic", "D3Q19", (150, 90, 110), 20, policy="FP64FP64",
              omega=1.7),
        # 16-bit block floating point on the 256^3 cavity
        _case("run_cavity_block_256", "run", "cavity", "D3Q19", (256, 256, 256), 40, policy="FP32I16_BLOCK"),
        # the wind tunnel: D3Q27, entropic collision, sphere, inlet, outlet, drag
        _case("run_tunnel_256x128x128", "run", "tunnel", "D3Q27", (256, 128, 128), 40, collision="KBC", omega=1.8),
        # gradients with respect to the initial state and the body force of the 2-D channel
        _case("rollout_channel2d_512x256", "rollout", "channel", "D2Q9", (512, 256), 60, omega=1.6),
        # gradients through a periodic turbulence box
        _case("rollout_periodic_128", "rollout", "periodic", "D3Q19", (128, 128, 128), 20, omega=1.8),
        # density, velocity, vorticity and Q-criterion of a 256^3 cavity
        _case("observe_cavity_256", "observe", "cavity", "D3Q19", (256, 256, 256), 0),
    ]


def _extents(rng, lo, hi, d, cells):
    """d extents between lo and hi, spread over their logarithm, with at most `cells` cells."""
    while True:
        e = [int(round(math.exp(rng.uniform(math.log(lo), math.log(hi))))) for _ in range(d)]
        if math.prod(e) <= cells:
            return tuple(e)


def draw(rng):
    omega = round(rng.uniform(0.8, 1.9), 3)
    what = rng.choice(["loop2d", "loop3d", "run2d", "run3d", "run3d", "run3d", "tunnel", "rollout2d", "rollout3d", "observe"])
    walls = rng.choice(["halfway", "fullway"])
    if what == "loop2d":
        return _case(None, "loop", "cavity", "D2Q9", _extents(rng, 24, 400, 2, 1 << 17), rng.randint(8, 24), omega=omega,
                     collision=rng.choice(["BGK", "BGK", "KBC"]), walls=walls)
    if what == "loop3d":
        lattice = rng.choice(["D3Q19", "D3Q27"])
        return _case(None, "loop", rng.choice(["cavity", "periodic"]), lattice, _extents(rng, 20, 200, 3, 1 << 21),
                     rng.randint(4, 12), omega=omega, walls=walls,
                     collision=rng.choice(["BGK", "SmagorinskyLESBGK"] + (["KBC"] if lattice == "D3Q27" else [])))
    if what == "run2d":
        flow = rng.choice(["channel", "cavity", "periodic"])
        return _case(None, "run", flow, "D2Q9", _extents(rng, 48, 2048, 2, 1 << 20), rng.randint(30, 120), omega=omega,
                     policy=rng.choice(["FP32FP32", "FP64FP64"]), walls=walls)
    if what == "run3d":
        policy = rng.choice(["FP32FP32", "FP32FP32", "FP32FP32", "FP64FP64", "FP32I16_BLOCK", "FP32FP16_SHIFTED",
                             "FP32FP32_DEVIATION"])
        shape = _extents(rng, 32, 512, 3, 1 << (23 if policy == "FP64FP64" else 24))
        lattice = "D3Q19" if policy == "FP32FP32_DEVIATION" else rng.choice(["D3Q19", "D3Q19", "D3Q27"])
        return _case(None, "run", rng.choice(["cavity", "periodic"]), lattice, shape, rng.randint(10, 24), policy=policy,
                     omega=omega, walls=walls)
    if what == "tunnel":
        lattice, collision = rng.choice([("D3Q19", "BGK"), ("D3Q27", "BGK"), ("D3Q27", "KBC")])
        return _case(None, "run", "tunnel", lattice, _extents(rng, 40, 200, 3, 1 << 22), rng.randint(10, 30), omega=omega,
                     collision=collision)
    if what == "rollout2d":
        return _case(None, "rollout", "channel", "D2Q9", _extents(rng, 48, 700, 2, 1 << 18), rng.randint(16, 60), omega=omega)
    if what == "rollout3d":
        lattice = rng.choice(["D3Q19", "D3Q19", "D3Q27"])
        return _case(None, "rollout", "periodic", lattice, _extents(rng, 24, 144, 3, 1 << 21), rng.randint(6, 20),
                     omega=omega, collision=rng.choice(["BGK", "SmagorinskyLESBGK"]))
    return _case(None, "observe", rng.choice(["cavity", "periodic"]), "D3Q19", _extents(rng, 40, 320, 3, 1 << 24), 0,
                 policy=rng.choice(["FP32FP32", "FP32FP32", "FP64FP64"]), walls=walls)


# ------------------------------------------------------------------------------------------------
# Inputs, from the seed alone
# ------------------------------------------------------------------------------------------------
def _device():
    return torch.device("cuda" if torch.cuda.is_available() else "cpu")


def _shape(case):
    return case["nx"], case["ny"], case["nz"]


def _waves(gen, shape, dev, count):
    """`count` smooth random float64 fields on `shape`: a few sine modes each, of unit scale."""
    axes = [torch.arange(n, dtype=torch.float64, device=dev) * (2 * math.pi / n) for n in shape]
    for _ in range(count):
        out = torch.zeros(shape, dtype=torch.float64, device=dev)
        for _ in range(3):
            k = torch.randint(1, 4, (3,), generator=gen).tolist()
            phase = (2 * math.pi * torch.rand(3, generator=gen, dtype=torch.float64)).tolist()
            s = [torch.sin(k[i] * axes[i] + phase[i]) if shape[i] > 1 else torch.ones_like(axes[i]) for i in range(3)]
            out += s[0].view(-1, 1, 1) * s[1].view(1, -1, 1) * s[2].view(1, 1, -1)
        yield out


def _initial(case, seed, dev):
    """rho (1, ...) and u (d, ...) of a smooth random flow, float64."""
    gen = torch.Generator().manual_seed(int(seed))
    d = 2 if case["lattice"] == "D2Q9" else 3
    fields = list(_waves(gen, _shape(case), dev, d + 1))
    return (1.0 + 1e-3 * fields[0]).unsqueeze(0), LID * torch.stack(fields[1:])


def _force(case, seed, dev):
    """The channel's body-force field (2, ...), float64."""
    gen = torch.Generator().manual_seed(int(seed) + 1)
    return 1e-5 * torch.stack(list(_waves(gen, _shape(case), dev, 2)))


def _cotangent(case, seed, dev, q):
    """dL/df at the end of a rollout (q, ...), float32: smooth in space, different in each direction."""
    gen = torch.Generator().manual_seed(int(seed) + 2)
    a, b = _waves(gen, _shape(case), dev, 2)
    m = torch.randn((2, q), generator=gen, dtype=torch.float64).to(dev).view(2, q, 1, 1, 1)
    return (m[0] * a + m[1] * b).float()


def _inlet_profile(ny):
    h = ny - 1.0
    return lambda y: 4.0 * 0.05 * y * (h - y) / (h * h)


INLET_3D = 0.04


def _sphere(case):
    """(centre, radius) of the tunnel's sphere: a tenth of the smallest cross extent."""
    nx, ny, nz = _shape(case)
    return (nx // 4, ny // 2, nz // 2), max(3.0, min(ny, nz) / 10.0)


def _in_sphere(case, dev):
    centre, r = _sphere(case)
    ax = [torch.arange(n, dtype=torch.float64, device=dev) - c for n, c in zip(_shape(case), centre)]
    return ax[0].view(-1, 1, 1) ** 2 + ax[1].view(1, -1, 1) ** 2 + ax[2].view(1, 1, -1) ** 2 < r * r


# ------------------------------------------------------------------------------------------------
# The framework's side
# ------------------------------------------------------------------------------------------------
def _walls(grid, names):
    """The cells of the named faces, each once, as index lists."""
    box = grid.bounding_box_indices()
    cells = torch.cat([torch.tensor(box[n]) for n in names], dim=1)
    return torch.unique(cells, dim=1).tolist()


def _boundary_conditions(case, grid):
    BC = xa.operator.boundary_condition
    flow = case["flow"]
    if flow == "periodic":
        return []
    inner = grid.bounding_box_indices(remove_edges=True)
    wall = BC.FullwayBounceBackBC if case["walls"] == "fullway" else BC.HalfwayBounceBackBC
    if flow == "cavity":
        two = case["lattice"] == "D2Q9"
        names = ["bottom", "left", "right"] + ([] if two else ["front", "back"])
        u = (LID, 0.0) if two else (LID, 0.0, 0.0)
        return [BC.EquilibriumBC(rho=1.0, u=u, indices=inner["top"]), wall(indices=_walls(grid, names))]
    if flow == "channel":
        profile = _inlet_profile(case["ny"])
        return [
            BC.HalfwayBounceBackBC(indices=_walls(grid, ["bottom", "top"])),
            BC.RegularizedBC("velocity", profile=lambda index: profile(index[1].astype(float)), indices=inner["left"]),
            BC.ExtrapolationOutflowBC(indices=inner["right"]),
        ]
    sphere = torch.nonzero(_in_sphere(case, torch.device("cpu"))).T.tolist()
    return [
        BC.FullwayBounceBackBC(indices=_walls(grid, ["bottom", "top", "front", "back"])),
        BC.RegularizedBC("velocity", prescribed_value=(INLET_3D, 0.0, 0.0), indices=inner["left"]),
        BC.ExtrapolationOutflowBC(indices=inner["right"]),
        BC.HalfwayBounceBackBC(indices=sphere),
    ]


def prepare(case, seed):
    dev = _device()
    policy = xa.PrecisionPolicy[case["policy"]]
    backend = xa.ComputeBackend.MI355X
    vs = getattr(xa.velocity_set, case["lattice"])(policy, backend)
    xa.init(velocity_set=vs, default_backend=backend, default_precision_policy=policy)
    xa.operator.boundary_condition.boundary_condition_registry.reset()
    shape = _shape(case)
    grid = xa.grid.grid_factory(shape[: vs.d], compute_backend=backend)
    bcs = _boundary_conditions(case, grid)
    compute = policy.compute_precision.torch_dtype
    force = _force(case, seed, dev).to(compute) if case["flow"] == "channel" else None
    stepper = xa.operator.stepper.IncompressibleNavierStokesStepper(grid, bcs, collision_type=case["collision"], force_field=force)
    f_0, f_1, bc_mask, missing_mask = stepper.prepare_fields()
    rho, u = _initial(case, seed, dev)
    if policy.block:
        xa.operator.equilibrium.QuadraticEquilibrium()(rho.to(compute), u.to(compute), f_0)
    else:
        f_0.copy_(_stored(case, rho, u, STORE[case["policy"]]))
    xa.grid.copy_population(f_1, f_0)
    state = dict(case=case, stepper=stepper, f_0=f_0, f_1=f_1, bc_mask=bc_mask, missing_mask=missing_mask)
    state["macroscopic"] = xa.operator.macroscopic.Macroscopic()
    state["rho"] = grid.create_field(1, dtype=policy.compute_precision)
    state["u"] = grid.create_field(vs.d, dtype=policy.compute_precision)
    if case["flow"] == "tunnel":
        state["drag"] = xa.operator.force.MomentumTransfer(bcs[3])
    if case["kind"] == "rollout":
        state["f_0"] = f_0.contiguous().requires_grad_()
        state["force"] = force.requires_grad_() if force is not None else None
        state["cotangent"] = _cotangent(case, seed, dev, vs.q)
    if case["kind"] == "observe":
        state["vorticity"] = xa.operator.postprocess.Vorticity()
        state["q_criterion"] = xa.operator.postprocess.QCriterion()
        state["fields"] = {n: grid.create_field(3 if n == "vorticity" else 1, dtype=policy.compute_precision)
                           for n in ("vorticity", "magnitude", "norm_mu", "q")}
    return state


def run(state):
    case, stepper = state["case"], state["stepper"]
    masks = state["bc_mask"], state["missing_mask"]
    f_0, f_1, omega, steps = state["f_0"], state["f_1"], case["omega"], case["steps"]
    if case["kind"] == "rollout":
        inputs = [f_0] + ([state["force"]] if state["force"] is not None else [])
        f = xa.autodiff.rollout(stepper, f_0, *masks, omega, steps, force_field=state["force"])
        return [f.detach()] + list(torch.autograd.grad(f, inputs, state["cotangent"]))
    if case["kind"] == "observe":
        rho, u = state["macroscopic"](f_0, state["rho"], state["u"])
        o = state["fields"]
        vort, mag = state["vorticity"](u, masks[0], o["vorticity"], o["magnitude"])
        mu, q = state["q_criterion"](u, masks[0], o["norm_mu"], o["q"])
        return dict(rho=rho, u=u, vorticity=vort, magnitude=mag, norm_mu=mu, q=q)
    if case["kind"] == "loop":
        for t in range(steps):
            f_0, f_1 = stepper(f_0, f_1, *masks, omega, t)
            f_0, f_1 = f_1, f_0
    else:
        f_0, f_1 = stepper.run(f_0, f_1, *masks, omega, steps)
    state["f_0"], state["f_1"] = f_0, f_1
    out = dict(f_0=f_0, f_1=f_1)
    if case["policy"] == "FP32I16_BLOCK":
        out["rho"], out["u"] = state["macroscopic"](f_0, state["rho"], state["u"])
    if case["flow"] == "tunnel":
        out["force"] = state["drag"].force_tensor(f_0, f_1, *masks)
    return out


def work(case):
    """Bytes: the state read and both buffers written (a rollout: the state, the cotangent and the
    force read, the final state and the gradients written; observe: the state and the ids read, ten
    fields written).  Operations: moments, equilibrium and relaxation of every cell update, about
    q (2 d + 12 + ...) each; a reverse step counts two forward ones besides the forward pass."""
    d, q = {"D2Q9": (2, 9), "D3Q19": (3, 19), "D3Q27": (3, 27)}[case["lattice"]]
    n = math.prod(_shape(case))
    size = torch.empty(0, dtype=STORE[case["policy"]]).element_size()
    ids = 0 if case["flow"] == "periodic" else n
    force = 2 * 4 * n if case["flow"] == "channel" else 0
    update = q * (4 * d + 9) * (2 if case["collision"] != "BGK" else 1)
    if case["kind"] == "observe":
        return {"bytes": n * q * size + 10 * n * max(size, 4) + ids, "flops": n * (q * (d + 1) + 60)}
    if case["kind"] == "rollout":
        return {"bytes": 4 * n * q * size + 2 * force + ids, "flops": 3 * n * update * case["steps"]}
    return {"bytes": 3 * n * q * size + force + ids, "flops": n * update * case["steps"]}


# ------------------------------------------------------------------------------------------------
# The same outputs in float64, by plain torch
# ------------------------------------------------------------------------------------------------
class _Lattice:
    def __init__(self, name):
        if name == "D2Q9":
            self.c = [(0, 0), (0, 1), (0, -1), (1, 0), (-1, 1), (1, -1), (-1, 0), (1, 1), (-1, -1)]
            weights = {0: 4 / 9, 1: 1 / 9, 2: 1 / 36}
        else:
            most = 2 if name == "D3Q19" else 3
            self.c = [c for c in itertools.product((0, -1, 1), repeat=3) if sum(map(abs, c)) <= most]
            weights = {0: 1 / 3, 1: 1 / 18, 2: 1 / 36} if most == 2 else {0: 8 / 27, 1: 2 / 27, 2: 1 / 54, 3: 1 / 216}
        self.d, self.q = len(self.c[0]), len(self.c)
        self.w = [weights[sum(map(abs, c))] for c in self.c]
        self.opp = [self.c.index(tuple(-v for v in c)) for c in self.c]

    def dot(self, l, u):
        return sum((c * u[i] for i, c in enumerate(self.c[l]) if c), 0.0)

    def feq(self, l, rho, u):
        cu = 3.0 * self.dot(l, u)
        return rho * self.w[l] * (1.0 + cu * (1.0 + 0.5 * cu) - 1.5 * sum(v * v for v in u))

    def moments(self, f):
        rho = sum(f)
        return rho, [sum(c[i] * f[l] for l, c in enumerate(self.c) if c[i]) / rho for i in range(self.d)]


def _stored(case, rho, u, dtype):
    """feq(rho, u) as the policy stores it."""
    lat = _Lattice(case["lattice"])
    shifted = case["policy"].endswith("_SHIFTED")
    return torch.stack([(lat.feq(l, rho[0], list(u)) - (lat.w[l] if shifted else 0.0)).to(dtype) for l in range(lat.q)])


def _collide(lat, f, collision, omega):
    rho, u = lat.moments(f)
    feq = [lat.feq(l, rho, u) for l in range(lat.q)]
    if collision == "BGK":
        return [a - omega * (a - e) for a, e in zip(f, feq)], rho, u
    neq = [a - e for a, e in zip(f, feq)]
    if collision == "SmagorinskyLESBGK":
        # the eddy viscosity from the directions of component sum 1 (once) and 2 or more (twice)
        strain = 0.0
        for l, c in enumerate(lat.c):
            if sum(c) >= 1:
                strain = strain + (1.0 if sum(c) == 1 else 2.0) * neq[l] ** 2
        t0 = 1.0 / omega
        tau = t0 + 0.5 * (torch.sqrt(t0 * t0 + 36.0 * SMAGORINSKY**2 * torch.sqrt(strain)) - t0)
        return [a - n / tau for a, n in zip(f, neq)], rho, u
    # KBC: the shear part relaxes with omega, the rest with the entropic stabiliser gamma
    pi = {(a, b): sum(c[a] * c[b] * neq[l] for l, c in enumerate(lat.c) if c[a] * c[b]) for a in range(lat.d) for b in range(a, lat.d)}
    shear = []
    for c in lat.c:
        axes = [i for i in range(lat.d) if c[i]]
        if len(axes) == 1 and lat.d == 3:
            shear.append(rho * (2 * pi[axes[0], axes[0]] - sum(pi[b, b] for b in range(3) if b != axes[0])) / 6.0)
        elif len(axes) == 1:
            shear.append(rho * (pi[axes[0], axes[0]] - pi[1 - axes[0], 1 - axes[0]]) / 4.0)
        elif len(axes) == 2:
            shear.append(rho * c[axes[0]] * c[axes[1]] * pi[axes[0], axes[1]] / 4.0)
        else:
            shear.append(torch.zeros_like(rho))
    sp1 = sp2 = 0.0
    for l in range(lat.q):
        high = neq[l] - shear[l]
        sp1 = sp1 + high * shear[l] / feq[l]
        sp2 = sp2 + high * high / feq[l]
    beta = 0.5 * omega
    gamma = 1.0 / beta - (2.0 - 1.0 / beta) * sp1 / (1e-32 + sp2)
    return [a - beta * (2.0 * s + gamma * (n - s)) for a, s, n in zip(f, shear, neq)], rho, u


class _Reference:
    """One step of a case in float64; fields are lists of q tensors (nx, ny, nz)."""

    def __init__(self, case, dev):
        self.case, self.lat, self.dev = case, _Lattice(case["lattice"]), dev
        lat, shape, flow = self.lat, _shape(case), case["flow"]
        self.shape = shape

        def face(axis, last, trim=0):
            m = torch.zeros(shape, dtype=torch.bool, device=dev)
            at = [slice(trim, n - trim) for n in shape[: lat.d]]
            at[axis] = shape[axis] - 1 if last else 0
            m[tuple(at)] = True
            return m

        self.outside = []  # cells whose source in direction l lies outside the domain
        for c in lat.c:
            m = torch.zeros(shape, dtype=torch.bool, device=dev)
            for i, v in enumerate(c):
                if v:
                    m |= face(i, v < 0)
            self.outside.append(m)
        none = torch.zeros(shape, dtype=torch.bool, device=dev)
        self.lid, self.fullway, self.halfway, self.inlet, self.outlet, self.body = none, none, none, none, none, none
        self.missing = self.outside
        if flow == "cavity":
            top = lat.d - 1
            self.lid = face(top, True, 1)
            # a later boundary condition takes the edges; the lid has none of them
            walls = face(top, False) | face(0, False) | face(0, True)
            if lat.d == 3:
                walls = walls | face(1, False) | face(1, True)
            if case["walls"] == "fullway":
                self.fullway = walls
            else:
                self.halfway = walls
        elif flow == "channel":
            self.halfway = face(1, False) | face(1, True)
            self.inlet, self.outlet = face(0, False, 1), face(0, True, 1)
        elif flow == "tunnel":
            self.fullway = face(1, False) | face(1, True) | face(2, False) | face(2, True)
            self.inlet, self.outlet = face(0, False, 1), face(0, True, 1)
            ball = _in_sphere(case, dev)
            pushed = [torch.roll(ball, c, (0, 1, 2)) for c in lat.c]
            self.body = torch.stack(pushed).any(0)
            self.halfway = self.body
            self.missing = [o | p for o, p in zip(self.outside, pushed)]
        self.ids = (self.lid | self.fullway | self.halfway | self.inlet | self.outlet) if flow != "periodic" else none
        if flow == "channel":
            speed = _inlet_profile(case["ny"])(torch.arange(1, shape[1] - 1, dtype=torch.float64, device=dev))
            self.speed = speed.to(STORE[case["policy"]]).double().view(1, -1, 1)
        elif flow == "tunnel":
            self.speed = float(torch.tensor(INLET_3D, dtype=STORE[case["policy"]]))

    def inlet_values(self, f):
        """The regularized velocity inlet on the inner cells of the plane x = 0."""
        lat = self.lat
        at = (slice(0, 1),) + tuple(slice(1, n - 1) for n in self.shape[1: lat.d])
        g = [a[at] for a in f]
        known = sum(g[l] for l, c in enumerate(lat.c) if c[0] < 0)
        rho = (2.0 * known + sum(g[l] for l, c in enumerate(lat.c) if c[0] == 0)) / (1.0 - self.speed)
        u = [self.speed + torch.zeros_like(rho)] + [torch.zeros_like(rho)] * (lat.d - 1)
        feq = [lat.feq(l, rho, u) for l in range(lat.q)]
        g = [g[lat.opp[l]] + feq[l] - feq[lat.opp[l]] if c[0] > 0 else g[l] for l, c in enumerate(lat.c)]
        out = []
        pi = {(a, b): sum(c[a] * c[b] * (g[l] - feq[l]) for l, c in enumerate(lat.c)) for a in range(lat.d) for b in range(lat.d)}
        for l, c in enumerate(lat.c):
            proj = sum((c[a] * c[b] - (1.0 / 3.0 if a == b else 0.0)) * pi[a, b] for a in range(lat.d) for b in range(lat.d))
            out.append(feq[l] + 4.5 * lat.w[l] * proj)
        new = []
        for l in range(lat.q):
            a = torch.zeros_like(f[l])
            a[at] = out[l]
            new.append(torch.where(self.inlet, a, f[l]))
        return new

    def step(self, f, omega, force=None):
        lat, dims = self.lat, tuple(range(self.lat.d))
        s = [torch.roll(f[l], c, dims) for l, c in enumerate(lat.c)]
        flow = self.case["flow"]
        if flow == "cavity":
            one = torch.ones((), dtype=torch.float64, device=self.dev)
            u = [LID * one] + [0.0 * one] * (lat.d - 1)
            s = [torch.where(self.lid, lat.feq(l, one, u), s[l]) for l in range(lat.q)]
        if flow != "periodic":
            bounce = self.halfway | self.outlet
            s = [torch.where(bounce & self.missing[l], f[lat.opp[l]], s[l]) for l in range(lat.q)]
        if flow in ("channel", "tunnel"):
            s = self.inlet_values(s)
        out, rho, u = _collide(lat, s, self.case["collision"], omega)
        if force is not None:
            uf = [u[i] + force[i] for i in range(lat.d)]
            out = [a + lat.feq(l, rho, uf) - lat.feq(l, rho, u) for l, a in enumerate(out)]
        if self.fullway.any():
            out = [torch.where(self.fullway, s[lat.opp[l]], out[l]) for l in range(lat.q)]
        if flow in ("channel", "tunnel"):
            # outgoing slots of the outlet hold the upwind value the next step's bounce-back reads
            cs = math.sqrt(1.0 / 3.0)
            for l, c in enumerate(lat.c):
                if c[0] < 0:
                    beside = torch.roll(f[l], (0,) + c[1:], dims)
                    o = lat.opp[l]
                    out[o] = torch.where(self.outlet & self.missing[l], (1.0 - cs) * f[o] + cs * beside, out[o])
        return out

    def drag(self, f):
        """Momentum exchange on the sphere: every missing population bounces back."""
        lat = self.lat
        cells = self.body & ~self.missing[0]
        total = [0.0] * lat.d
        for l in range(lat.q):
            o = lat.opp[l]
            both = (2.0 * f[o] * (cells & self.missing[l])).sum()
            for i in range(lat.d):
                total[i] = total[i] + lat.c[o][i] * both
        return torch.stack(total)


def _exact_observe(case, ref, f):
    rho, u = ref.lat.moments(f)

    def d(a, axis):
        return (torch.roll(a, -1, axis) - torch.roll(a, 1, axis)) / 2.0

    g = [[d(u[i], j) for j in range(3)] for i in range(3)]
    near = torch.zeros_like(ref.ids)
    for axis, way in itertools.product(range(3), (1, -1)):
        near |= torch.roll(ref.ids, way, axis)
    keep = torch.zeros_like(near)
    keep[1:-1, 1:-1, 1:-1] = True
    keep &= ~near
    curl = [g[2][1] - g[1][2], g[0][2] - g[2][0], g[1][0] - g[0][1]]
    curl = [torch.where(keep, v, 0.0) for v in curl]
    mag = torch.sqrt(sum(v * v for v in curl)).unsqueeze(0)
    # (|antisymmetric part|^2 - |symmetric part|^2) / 2 of the velocity gradient
    q = -0.5 * sum(g[i][j] * g[j][i] for i in range(3) for j in range(3))
    q = torch.where(keep, q, 0.0).unsqueeze(0)
    return dict(rho=rho.unsqueeze(0), u=torch.stack(u), vorticity=torch.stack(curl), magnitude=mag, norm_mu=mag, q=q)


def exact(case, seed):
    dev = _device()
    ref = _Reference(case, dev)
    lat, omega, steps = ref.lat, case["omega"], case["steps"]
    block = case["policy"] == "FP32I16_BLOCK"
    store = torch.float64 if block else STORE[case["policy"]]
    rho, u = _initial(case, seed, dev)
    if block:
        rho, u = rho.float().double(), u.float().double()
    f = _stored(case, rho, u, store).double()
    shift = torch.tensor(lat.w, dtype=torch.float64, device=dev).view(-1, 1, 1, 1) if case["policy"].endswith("_SHIFTED") else None
    if shift is not None:
        f = f + shift
    force = None
    if case["flow"] == "channel":
        force = _force(case, seed, dev)
        force = force if case["policy"] == "FP64FP64" else force.float().double()
    if case["kind"] == "observe":
        return _exact_observe(case, ref, list(f))
    if case["kind"] == "rollout":
        inputs = [f.requires_grad_()] + ([force.requires_grad_()] if force is not None else [])

        def advance(state, *g):
            return torch.stack(ref.step(list(state), omega, g[0] if g else None))

        out = f
        for _ in range(steps):
            out = checkpoint(advance, out, *inputs[1:], use_reentrant=False)
        return [out.detach()] + list(torch.autograd.grad(out, inputs, _cotangent(case, seed, dev, lat.q).double()))
    f, last = list(f), None
    for _ in range(steps):
        last, f = f, ref.step(f, omega, force)

    def laid(g):
        if block:
            return None
        g = torch.stack(g)
        return g - shift if shift is not None else g

    out = dict(f_0=laid(f), f_1=laid(last))
    if block:
        rho, u = lat.moments(f)
        out["rho"], out["u"] = rho.unsqueeze(0), torch.stack(u)
    if case["flow"] == "tunnel":
        out["force"] = ref.drag(f)
    return out
