"""The work that a program does with this framework, as cases to time and to compare.

listed() names the cases, draw() gives further ones of the same ranges, prepare() builds what a
program holds before the call (lattice, boundary lists, fields, drivers), run() is one pass
through the public entry points, work() the bytes and operations of a pass and exact() its result
in 64 bits, from plain torch formulas below.

Kinds of case:
  box             time steps of a periodic box (Simulation.run): homogeneous flow, Taylor-Green
  cavity          time steps of a lid-driven cavity, bounce-back walls and lid
  sphere          time steps of a channel flow past a sphere (velocity inflow, pressure outlet,
                  interpolated walls and sphere, Brinkman porosity), the drag read between runs
  sparse          the same flow on the neighbour-list layout (box=False), as a level that is not a
                  dense box is stepped
  sphere_grad     forward and backward through k17_steps: the drag's gradient in the porosity
  two_level       coarse steps of a channel with a refined box (MultiLevelSimulation.run)
  two_level_grad  forward and backward through k17_two_level_steps: the flow energy's gradient in the
                  inflow's amplitudes and the porosity of the refined box
  monitor         the analysis between two output intervals: FP64 moment sums, macroscopic fields and
                  kinetic energy of one state
"""
import functools
import math
import types

import numpy as np
import torch
from torch.utils.checkpoint import checkpoint

from virtualfluids_amd import adjoint
from virtualfluids_amd.grid import Grid, channel, d0M0, d0P0, d00M, d00P, dM00, dP00, sphere_channel, walled_box
from virtualfluids_amd.lattice import Lattice
from virtualfluids_amd.refinement import GridScalingFactory, nested_box
from virtualfluids_amd.simulation import BoundaryConditionFactory, MultiLevelSimulation, Simulation

DTYPE = {"fp32": torch.float32, "fp16": torch.float16, "bf16": torch.bfloat16}
FLOPS_PER_NODE = 1000          # collision: about 690 vector operations, half of them fused
FLOPS_PER_NODE_ADJOINT = 2500  # its reverse, with the forward part it recomputes
LIMITER = 0.01
INFLOW = 0.04


# ---- the cases --------------------------------------------------------------------------------
def listed():
    return [
        # the smallest lattice that a user steps, in a long run: launches and latency count
        {"name": "cavity_32", "kind": "cavity", "n": 32, "storage": "fp32", "omega": 1.8, "steps": 1000},
        # the reference's published GPU benchmark, 64 nodes a side
        {"name": "cavity_64", "kind": "cavity", "n": 64, "storage": "fp32", "omega": 1.8, "steps": 500},
        # Taylor-Green 256^3, the framework's default benchmark, in the storage types it offers
        {"name": "box_256_fp32", "kind": "box", "nx": 256, "ny": 256, "nz": 256, "storage": "fp32", "omega": 1.95,
         "steps": 20},
        {"name": "box_256_fp16", "kind": "box", "nx": 256, "ny": 256, "nz": 256, "storage": "fp16", "omega": 1.95,
         "steps": 20},
        # the largest benchmark size
        {"name": "box_512_fp32", "kind": "box", "nx": 512, "ny": 512, "nz": 512, "storage": "fp32", "omega": 1.97,
         "steps": 4},
        # a box whose extents nobody chose for the hardware
        {"name": "box_odd_bf16", "kind": "box", "nx": 251, "ny": 187, "nz": 133, "storage": "bf16", "omega": 1.9,
         "steps": 40},
        # flow past a sphere at the benchmark's size, the drag read every 100 steps
        {"name": "sphere", "kind": "sphere", "nx": 192, "ny": 96, "nz": 96, "storage": "fp32", "omega": 1.8,
         "steps": 100, "rounds": 2},
        # the neighbour-list layout of the reference's data contract
        {"name": "sparse", "kind": "sparse", "nx": 192, "ny": 96, "nz": 96, "storage": "fp32", "omega": 1.8,
         "steps": 40},
        # inverse problem on the sphere channel: checkpointed forward, replay and adjoint
        {"name": "sphere_grad", "kind": "sphere_grad", "nx": 192, "ny": 96, "nz": 96, "storage": "fp32",
         "omega": 1.8, "steps": 100, "every": 50},
        # channel with a 2:1 refined box at the benchmark's size, 16-bit storage
        {"name": "two_level", "kind": "two_level", "nx": 256, "ny": 128, "nz": 128, "storage": "fp16",
         "omega": 1.91, "steps": 50},
        # its gradient, the benchmark's optimisation of the inflow profile
        {"name": "two_level_grad", "kind": "two_level_grad", "nx": 256, "ny": 128, "nz": 128, "storage": "fp16",
         "omega": 1.91, "steps": 40, "every": 20},
        # what a monitored run computes at each output interval
        {"name": "monitor_256", "kind": "monitor", "nx": 256, "ny": 256, "nz": 256, "storage": "fp32", "omega": 1.95},
    ]


def draw(rng):
    """One more case: sizes spread over their range (by their logarithm), odd ones among them."""
    def size(lo, hi, step=1):
        return max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi))) / step)) * step)

    kind = rng.choice(["box", "box", "box", "cavity", "sphere", "sparse", "sphere_grad", "two_level",
                       "two_level_grad", "monitor"])
    case = {"kind": kind, "storage": rng.choice(["fp32", "fp16", "bf16"]), "omega": round(rng.uniform(1.78, 1.96), 4)}
    if kind in ("box", "monitor"):
        step = rng.choice([1, 1, 2, 64])  # ragged rows, and rows of whole waves
        case.update(nx=size(64 if step == 64 else 33, 384, step), ny=size(24, 320), nz=size(24, 320))
        if kind == "box":
            case["steps"] = rng.choice([2, 5, 10, 20])
    elif kind == "cavity":
        case.update(n=size(16, 96), storage="fp32", steps=rng.choice([100, 333, 400]))
    elif kind in ("sphere", "sparse", "sphere_grad"):
        ny = size(32, 104, 2)
        case.update(nx=size(64, 230, 2), ny=ny, nz=max(32, ny - rng.choice([0, 3, 8])),
                    steps=rng.choice([21, 40, 60]))
        if kind == "sphere":
            case["rounds"] = rng.choice([1, 2])
        if kind == "sphere_grad":
            case["every"] = rng.choice([7, 10, 20])
    else:
        case.update(nx=size(64, 256, 4), ny=size(48, 128, 4), nz=size(48, 128, 4), steps=rng.choice([12, 20, 30]),
                    omega=round(rng.uniform(1.88, 1.95), 4))
        if kind == "two_level_grad":
            case["every"] = rng.choice([5, 6, 10])
    return case


# ---- grids (host arrays; a program builds them once) ------------------------------------------
@functools.lru_cache(maxsize=4)
def _box_grid(nx, ny, nz):
    n = np.arange(nx * ny * nz, dtype=np.uint32)
    k = n.reshape(nz, ny, nx)
    nb = [np.ascontiguousarray(np.roll(k, -1, axis)).ravel() for axis in (2, 1, 0)]
    return Grid(nx, ny, nz, *nb, np.full(n.size, 19, dtype=np.uint32), n)


@functools.lru_cache(maxsize=4)
def _cavity_grid(n):
    walls = {s: ("noslip",) for s in (dP00, dM00, d0P0, d0M0, d00M)}
    walls[d00P] = ("velocity", (0.05 / math.sqrt(2.0), 0.05 / math.sqrt(2.0), 0.0))
    return walled_box((n, n, n), walls)


@functools.lru_cache(maxsize=4)
def _sphere_grid(nx, ny, nz):
    return sphere_channel((nx, ny, nz), (nx // 4, ny // 2, nz // 2), min(ny, nz) / 8.0, INFLOW)


@functools.lru_cache(maxsize=2)
def _nested(nx, ny, nz):
    lo = (nx // 4 + 1, ny // 4 + 1, nz // 4 + 1)
    hi = (nx // 2 + 1, 3 * ny // 4 + 1, 3 * nz // 4 + 1)
    return nested_box(None, lo, hi, coarse=channel((nx, ny, nz), inflow=0.03))


def _grid(case):
    if case["kind"] == "cavity":
        return _cavity_grid(case["n"])
    size = (case["nx"], case["ny"], case["nz"])
    if case["kind"] in ("box", "monitor"):
        return _box_grid(*size)
    return _sphere_grid(*size)


def _fine_omega(omega):
    """Relaxation rate one level finer: twice the viscosity in lattice units."""
    return 1.0 / (2.0 * (1.0 / omega - 0.5) + 0.5)


# ---- inputs -----------------------------------------------------------------------------------
def _mesh(grid, device="cuda"):
    return torch.meshgrid(*(torch.arange(n, device=device, dtype=torch.float32) for n in (grid.nz, grid.ny, grid.nx)),
                          indexing="ij")


def _populations(grid, storage, seed, mean, amplitude):
    """A flow state as a 27 N buffer (even parity): a Taylor-Green vortex of random phase on a mean
    flow in x, at equilibrium up to small random deviations; zero on solid nodes."""
    cpu = torch.Generator().manual_seed(int(seed))
    gpu = torch.Generator(device="cuda").manual_seed(int(seed))
    phase = 2 * math.pi * torch.rand(3, generator=cpu)
    drift = amplitude * 0.2 * (torch.rand(3, generator=cpu) - 0.5)
    z, y, x = _mesh(grid)
    x, y, z = (2 * math.pi / n * a + float(p) for n, a, p in zip((grid.nx, grid.ny, grid.nz), (x, y, z), phase))
    fluid = None
    if grid.fluid.size != grid.N:
        fluid = torch.from_numpy(grid.geo == 19).cuda().reshape(grid.nz, grid.ny, grid.nx)
    u = [mean + float(drift[0]) + amplitude * torch.sin(x) * torch.cos(y) * torch.cos(z),
         float(drift[1]) - amplitude * torch.cos(x) * torch.sin(y) * torch.cos(z),
         float(drift[2]) * torch.cos(x)]
    drho = 3.0 * amplitude ** 2 / 16.0 * (torch.cos(2 * x) + torch.cos(2 * y)) * (torch.cos(2 * z) + 2.0)
    del x, y, z
    usq = 1.5 * sum(a * a for a in u)
    out = torch.empty((27, grid.nz, grid.ny, grid.nx), dtype=DTYPE[storage], device="cuda")
    for d, c in enumerate(C):
        cu = 3.0 * sum(ci * ui for ci, ui in zip(c, u) if ci) + 0.0 * usq
        f = W[d] * (drho + (1.0 + drho) * (cu + 0.5 * cu * cu - usq))
        f += W[d] * 1e-4 * torch.randn(f.shape, generator=gpu, device="cuda")
        if fluid is not None:
            f = torch.where(fluid, f, 0.0)
        out[d] = _rolled(f, c, +1)
    return out.reshape(-1)


def _porosity(grid, seed, high=0.1, radius=None):
    """A smooth porosity field in [0, high], inside a ball around the centre where radius is given."""
    cpu = torch.Generator().manual_seed(int(seed) + 7)
    phase = 2 * math.pi * torch.rand(3, generator=cpu)
    z, y, x = _mesh(grid)
    field = high * 0.125 * (1 + torch.sin(x / 8 + float(phase[0]))) * (1 + torch.sin(y / 8 + float(phase[1]))) * (
        1 + torch.sin(z / 8 + float(phase[2])))
    if radius is not None:
        r2 = (x - grid.nx / 2) ** 2 + (y - grid.ny / 2) ** 2 + (z - grid.nz / 2) ** 2
        field = torch.where(r2 <= radius * radius, field, 0.0)
    return field.reshape(-1).contiguous()


def _inputs(case, seed):
    """The values a pass works on, made from the seed alone."""
    s = types.SimpleNamespace()
    if case["kind"] in ("two_level", "two_level_grad"):
        nb = _nested(case["nx"], case["ny"], case["nz"])
        s.f = [_populations(g, case["storage"], seed + i, 0.03, 0.005) for i, g in enumerate((nb.coarse, nb.fine))]
        s.porosity = _porosity(nb.fine, seed, radius=0.3 * min(nb.fine.nx, nb.fine.ny, nb.fine.nz))
        # inflow profile: sine modes over the inlet, near the series of a uniform flow
        vel = nb.coarse.bcs["velocity"]
        _, y, z = nb.coarse.coords()
        yh, zh = (y[vel.k] - 0.5) / case["ny"], (z[vel.k] - 0.5) / case["nz"]
        modes = [(m, n) for m in range(1, 9) for n in range(1, 5)]
        basis = np.stack([np.sin(m * np.pi * yh) * np.sin(n * np.pi * zh) for m, n in modes])
        s.basis = torch.from_numpy(basis.astype(np.float32)).cuda()
        a = np.array([0.03 * 16 / (np.pi ** 2 * m * n) if m % 2 and n % 2 else 0.0 for m, n in modes])
        a = a * (1.0 + 0.05 * np.random.RandomState(seed % (1 << 31)).standard_normal(a.size))
        s.amplitudes = torch.from_numpy(a.astype(np.float32)).cuda()
        return s
    grid = _grid(case)
    mean, amplitude = {"cavity": (0.0, 0.01), "box": (0.0, 0.05), "monitor": (0.02, 0.05)}.get(
        case["kind"], (INFLOW, 0.008))
    s.f = _populations(grid, case["storage"], seed, mean, amplitude)
    s.porosity = _porosity(grid, seed) if case["kind"] in ("sphere", "sparse", "sphere_grad") else None
    return s


# ---- what a program holds, and one pass -------------------------------------------------------
def _factory(kind):
    F = BoundaryConditionFactory
    fac = F()
    if kind == "cavity":
        fac.set_velocity_boundary_condition(F.VelocityBC.VelocityBounceBack)
        fac.set_no_slip_boundary_condition(F.NoSlipBC.NoSlipBounceBack)
    else:
        fac.set_velocity_boundary_condition(F.VelocityBC.VelocityInterpolatedCompressible)
        fac.set_no_slip_boundary_condition(F.NoSlipBC.NoSlipInterpolatedCompressible)
        fac.set_geometry_boundary_condition(F.NoSlipBC.NoSlipInterpolatedCompressible)
        fac.set_pressure_boundary_condition(F.PressureBC.PressureNonEquilibriumCompressible)
    return fac


def prepare(case, seed):
    kind = case["kind"]
    s = _inputs(case, seed)
    s.case = case
    limiters = (LIMITER,) * 3
    if kind in ("two_level", "two_level_grad"):
        nb = _nested(case["nx"], case["ny"], case["nz"])
        s.interface = (nb.cf, nb.fc)
        s.levels = [Lattice(g, om, storage=case["storage"], limiters=limiters, level=i)
                    for i, (g, om) in enumerate(((nb.coarse, case["omega"]), (nb.fine, _fine_omega(case["omega"]))))]
        s.factory = _factory(kind)
        if kind == "two_level":
            for L, f in zip(s.levels, s.f):
                L.f.copy_(f)
            ux = s.amplitudes @ s.basis
            s.levels[0].bcs["velocity"].vel[0].copy_(ux)
            s.levels[1].set_porosity(s.porosity)
            scaling = GridScalingFactory()
            scaling.set_scaling_factory(GridScalingFactory.GridScaling.ScaleCompressible)
            s.sim = MultiLevelSimulation(s.levels, [s.interface], [s.factory, None], scaling)
        else:
            s.observe = adjoint.KineticEnergyObservation(nb.coarse, _observed(nb))
        return s
    grid = _grid(case)
    s.lattice = Lattice(grid, case["omega"], storage=case["storage"], limiters=limiters, box=kind != "sparse")
    if kind == "sphere_grad":
        s.factory = _factory(kind)
        s.observe = adjoint.MomentumExchangeObservation(grid, "geometry", axis=0, scale=1.0 / case["steps"])
        return s
    s.lattice.f.copy_(s.f)
    s.f = None
    if s.porosity is not None:
        s.lattice.set_porosity(s.porosity)
    if kind == "monitor":
        s.lattice.moment_sums()  # as at the run's start
    else:
        s.sim = Simulation(s.lattice, None if kind == "box" else _factory(kind))
    return s


def run(s):
    case, kind = s.case, s.case["kind"]
    if kind in ("box", "cavity", "sparse"):
        s.sim.run(case["steps"])
        return {"populations": s.lattice.f}
    if kind == "sphere":
        drag = []
        for _ in range(case["rounds"]):
            s.sim.run(case["steps"])
            drag.append(s.lattice.drag_force("geometry"))
        return {"populations": s.lattice.f, "drag": np.stack(drag)}
    if kind == "two_level":
        s.sim.run(case["steps"])
        return {"coarse": s.levels[0].f, "fine": s.levels[1].f}
    if kind == "monitor":
        L = s.lattice
        sums = L.moment_sums()
        energy, nodes = L.kinetic_energy()
        return {"sums": sums, "energy": energy, "nodes": nodes, "rho": L.rho, "vx": L.vx, "vy": L.vy, "vz": L.vz,
                "pressure": L.press}
    if kind == "sphere_grad":
        phi = s.porosity.detach().clone().requires_grad_(True)
        f, J = adjoint.k17_steps(s.f, s.lattice, case["steps"], checkpoint_every=case["every"], even=True,
                                 bc_factory=s.factory, porosity=phi, observe=s.observe,
                                 observe_from=case["steps"] // 2)
        J.backward()
        return {"populations": f.detach(), "objective": J.detach().float(), "porosity_grad": phi.grad}
    a = s.amplitudes.detach().clone().requires_grad_(True)
    phi = s.porosity.detach().clone().requires_grad_(True)
    ux = a @ s.basis
    zero = torch.zeros_like(ux)
    fc, ff, J = adjoint.k17_two_level_steps(
        s.f[0], s.f[1], s.levels[0], s.levels[1], s.interface, case["steps"], checkpoint_every=case["every"], even=True,
        bc_factory=s.factory, velocity=torch.stack([ux, zero, zero]), porosity_fine=phi, observe=s.observe,
        observe_from=case["steps"] // 2)
    J.backward()
    return {"coarse": fc.detach(), "fine": ff.detach(), "objective": J.detach().float(), "amplitude_grad": a.grad,
            "porosity_grad": phi.grad}


def _observed(nb):
    """Coarse nodes whose energy is the objective: a plane behind the inflow and the shell on which
    the refined box hands its flow back."""
    x, _, _ = _coords(nb.coarse.nx, nb.coarse.ny, nb.coarse.nz)
    plane = np.nonzero((x == 4) & (nb.coarse.geo == 19))[0]
    return np.concatenate([plane, np.asarray(nb.fc.coarse, dtype=np.int64)])


def work(case):
    """Bytes and operations of a pass: every population of a node read and written once a step (and
    its reverse: the state read, the adjoint read and written, on top of one replayed step)."""
    e = DTYPE[case["storage"]].itemsize
    steps = case.get("steps", 1) * case.get("rounds", 1)
    if case["kind"] in ("two_level", "two_level_grad"):
        nx, ny, nz = case["nx"], case["ny"], case["nz"]
        coarse, fine = nx * ny * nz, 8 * (nx // 4) * (ny // 2) * (nz // 2)
        n = (coarse + 2 * fine) * steps
    elif case["kind"] == "cavity":
        n = case["n"] ** 3 * steps
    else:
        n = case["nx"] * case["ny"] * case["nz"] * steps
    if case["kind"] == "monitor":
        # populations and node types in, five fields out, the fields in again for the energy
        return {"bytes": n * (27 * e + 4 + 5 * 4 + 4 * 4), "flops": n * 200}
    if case["kind"] == "sparse":
        return {"bytes": n * (2 * 27 * e + 4 + 3 * 4 + 4), "flops": n * FLOPS_PER_NODE}
    if case["kind"].endswith("_grad"):
        return {"bytes": n * (4 * 27 * e + 27 * (e + 8) + 12), "flops": n * (2 * FLOPS_PER_NODE + FLOPS_PER_NODE_ADJOINT)}
    return {"bytes": n * 2 * 27 * e, "flops": n * FLOPS_PER_NODE}


# ---- the same in 64 bits, from the formulas ---------------------------------------------------
# D3Q27 velocities, opposites and weights in the order of the data contract
C = [(0, 0, 0), (1, 0, 0), (-1, 0, 0), (0, 1, 0), (0, -1, 0), (0, 0, 1), (0, 0, -1), (1, 1, 0), (-1, -1, 0),
     (1, -1, 0), (-1, 1, 0), (1, 0, 1), (-1, 0, -1), (1, 0, -1), (-1, 0, 1), (0, 1, 1), (0, -1, -1), (0, 1, -1),
     (0, -1, 1), (1, 1, 1), (-1, 1, 1), (1, -1, 1), (-1, -1, 1), (1, 1, -1), (-1, 1, -1), (1, -1, -1), (-1, -1, -1)]
OPPOSITE = [C.index((-a, -b, -c)) for a, b, c in C]
W = [(8 / 27, 2 / 27, 1 / 54, 1 / 216)[abs(a) + abs(b) + abs(c)] for a, b, c in C]


def _rolled(f, c, sign):
    """The population array f (nz, ny, nx) of direction c between the node that holds it and the
    cell that stores it (one further along every axis where c is negative): sign +1 to the cell,
    -1 back to the node."""
    shifts = [(sign, 2 - axis) for axis in range(3) if c[axis] < 0]
    return torch.roll(f, [s for s, _ in shifts], [a for _, a in shifts]) if shifts else f


def _pre_of_buffer(buf, grid, even):
    b = buf.reshape(27, grid.nz, grid.ny, grid.nx)
    out = torch.empty((27, grid.N), dtype=torch.float64, device=buf.device)
    for d in range(27):
        out[d] = _rolled(b[d if even else OPPOSITE[d]].double(), C[d], -1).reshape(-1)
    return out


def _buffer_of_pre(pre, grid, even):
    p = pre.reshape(27, grid.nz, grid.ny, grid.nx)
    out = torch.empty_like(p)
    for d in range(27):
        out[d if even else OPPOSITE[d]] = _rolled(p[d], C[d], +1)
    return out.reshape(-1)


def _streamed(post, grid):
    p = post.reshape(27, grid.nz, grid.ny, grid.nx)
    out = torch.empty_like(p)
    for d in range(27):
        out[d] = torch.roll(p[d], (C[d][2], C[d][1], C[d][0]), (0, 1, 2))
    return out.reshape(27, -1)


_CUBE = [C.index((i - 1, j - 1, k - 1)) for i in range(3) for j in range(3) for k in range(3)]


def _cube(f):
    """(27, n) shifted populations as (3, 3, 3, n) whole ones, index = velocity + 1 per axis."""
    w = torch.tensor(W, dtype=f.dtype, device=f.device)
    return (f + w[:, None])[_CUBE].reshape(3, 3, 3, -1)


def _list(cube):
    flat = cube.reshape(27, -1)
    order = [_CUBE.index(d) for d in range(27)]
    return flat[order] - torch.tensor(W, dtype=cube.dtype, device=cube.device)[:, None]


def _to_central(F, u):
    for axis in range(3):
        a, b, c = F.unbind(axis)
        s, d, e, v = a + b + c, c - a, a + c, u[axis]
        F = torch.stack([s, d - v * s, e - 2 * v * d + v * v * s], axis)
    return F


def _from_central(M, u):
    for axis in range(3):
        m0, m1, m2 = M.unbind(axis)
        v = u[axis]
        r1, r2 = m1 + v * m0, m2 + 2 * v * m1 + v * v * m0
        M = torch.stack([0.5 * (r2 - r1), m0 - r2, 0.5 * (r2 + r1)], axis)
    return M


def _rest_moments(m):
    """Adds the moments of the weights to the shifted moments {(a, b, c): value}."""
    rest = {0: 1.0, 2: 1.0 / 3.0}
    cube = []
    for i in range(27):
        a, b, c = i // 9, i // 3 % 3, i % 3
        w = rest.get(a, 0.0) * rest.get(b, 0.0) * rest.get(c, 0.0)
        cube.append(m[a, b, c] + w)
    return torch.stack(cube).reshape(3, 3, 3, -1)


def _collide(f, omega, phi=None):
    """K17 cumulant collision of (27, n) shifted populations (Geier et al. 2017,
    10.1016/j.jcp.2017.05.040), velocity scaled by 1 - phi / 2."""
    w = omega
    F = _cube(f)
    drho = f.sum(0)
    rho = 1.0 + drho
    c = torch.tensor(C, dtype=f.dtype, device=f.device)
    u = (c.T @ f) / rho
    if phi is not None:
        u = u * (1.0 - 0.5 * phi)
    M = _to_central(F, u)

    def m(a, b, c_):
        v = M[a, b, c_]
        if a % 2 == 0 and b % 2 == 0 and c_ % 2 == 0:
            v = v - (1.0 / 3.0) ** ((a + b + c_) // 2)
        return v

    m0 = m(0, 0, 0)
    p2, xy, xz = m(2, 0, 0) + m(0, 2, 0) + m(0, 0, 2), m(2, 0, 0) - m(0, 2, 0), m(2, 0, 0) - m(0, 0, 2)
    dx = -0.5 * w * (xy + xz) + 0.5 * (m0 - p2)
    dy, dz = dx + 1.5 * w * xy, dx + 1.5 * w * xz
    ux, uy, uz = (u[i] ** 2 * g for i, g in enumerate((dx, dy, dz)))
    trace = m0 - 1.5 * (ux + uy + uz)
    xy = (1 - w) * xy - 3 * (1 - 0.5 * w) * (ux - uy)
    xz = (1 - w) * xz - 3 * (1 - 0.5 * w) * (ux - uz)
    n = {(0, 0, 0): m0, (1, 0, 0): -m(1, 0, 0), (0, 1, 0): -m(0, 1, 0), (0, 0, 1): -m(0, 0, 1),
         (2, 0, 0): (xy + xz + trace) / 3, (0, 2, 0): (-2 * xy + xz + trace) / 3,
         (0, 0, 2): (xy - 2 * xz + trace) / 3,
         (1, 1, 0): (1 - w) * m(1, 1, 0), (1, 0, 1): (1 - w) * m(1, 0, 1), (0, 1, 1): (1 - w) * m(0, 1, 1)}
    # third order, rates limited
    plus = 8 * (w - 2) * (1 + 2 * w) / (7 * w * w - 14 * w - 8)
    minus = 8 * (w - 2) * (4 * w - 7) / (56 - 50 * w + 9 * w * w)
    triple = 24 * (w - 2) * (3 * w * w - 7 * w - 2) / (48 + 152 * w - 130 * w * w + 29 * w ** 3)

    def relaxed(x, rate):
        return x - x * (rate + (1 - rate) * x.abs() / (x.abs() + LIMITER))

    n[1, 1, 1] = relaxed(m(1, 1, 1), triple)
    for p, q in (((2, 1, 0), (0, 1, 2)), ((2, 0, 1), (0, 2, 1)), ((1, 2, 0), (1, 0, 2))):
        s, d = relaxed(m(*p) + m(*q), plus), relaxed(m(*p) - m(*q), minus)
        n[p], n[q] = 0.5 * (s + d), 0.5 * (s - d)
    # fourth order
    A = (4 + 2 * w - 3 * w * w) / (2 - 7 * w + 5 * w * w)
    B = (4 + 28 * w - 14 * w * w) / (6 - 21 * w + 15 * w * w)
    nu = 1 / w - 0.5
    n200, n020, n002, n110, n101, n011, n111 = (n[i] for i in (
        (2, 0, 0), (0, 2, 0), (0, 0, 2), (1, 1, 0), (1, 0, 1), (0, 1, 1), (1, 1, 1)))
    n[2, 1, 1] = nu * B * w * m(0, 1, 1) + ((n200 + 1 / 3) * n011 + 2 * n110 * n101) / rho
    n[1, 2, 1] = nu * B * w * m(1, 0, 1) + ((n020 + 1 / 3) * n101 + 2 * n110 * n011) / rho
    n[1, 1, 2] = nu * B * w * m(1, 1, 0) + ((n002 + 1 / 3) * n110 + 2 * n101 * n011) / rho
    for i, a, b, off, g in (((2, 2, 0), n200, n020, n110, dx + dy), ((2, 0, 2), n200, n002, n101, dx + dz),
                            ((0, 2, 2), n002, n020, n011, dy + dz)):
        n[i] = -nu * 2 / 3 * A * g + (a * b + 2 * off * off + (a + b) / 3 - drho / 9) / rho
    # fifth order: cumulants zero
    n210, n012, n201, n021, n120, n102 = (n[i] for i in ((2, 1, 0), (0, 1, 2), (2, 0, 1), (0, 2, 1), (1, 2, 0), (1, 0, 2)))
    n[1, 2, 2] = (n002 * n120 + n020 * n102 + 4 * n011 * n111 + 2 * (n101 * n021 + n110 * n012) + (n120 + n102) / 3) / rho
    n[2, 1, 2] = (n002 * n210 + n200 * n012 + 4 * n101 * n111 + 2 * (n011 * n201 + n110 * n102) + (n210 + n012) / 3) / rho
    n[2, 2, 1] = (n200 * n021 + n020 * n201 + 4 * n110 * n111 + 2 * (n101 * n120 + n011 * n210) + (n021 + n201) / 3) / rho
    # sixth order: cumulant zero
    n220, n202, n022, n211, n121, n112 = (n[i] for i in ((2, 2, 0), (2, 0, 2), (0, 2, 2), (2, 1, 1), (1, 2, 1), (1, 1, 2)))
    tr = n200 + n020 + n002
    t1 = (4 * n111 ** 2 + n200 * n022 + n020 * n202 + n002 * n220 + 4 * (n011 * n211 + n101 * n121 + n110 * n112)
          + 2 * (n120 * n102 + n210 * n012 + n201 * n021) + (n022 + n202 + n220) / 3 + tr / 9)
    t2 = (4 * (n101 ** 2 * n020 + n011 ** 2 * n200 + n110 ** 2 * n002) + 2 * n200 * n020 * n002 + 16 * n110 * n101 * n011
          + 2 / 3 * (2 * (n101 ** 2 + n011 ** 2 + n110 ** 2) + n002 * n020 + n002 * n200 + n020 * n200 + tr / 3)
          + (drho * drho - drho) / 27)
    n[2, 2, 2] = (t1 - t2 / rho) / rho
    return _list(_from_central(_rest_moments(n), u))


def _flow_moments(f):
    """Density deviation and velocity of (27, n) shifted populations."""
    drho = f.sum(0)
    return drho, (torch.tensor(C, dtype=f.dtype, device=f.device).T @ f) / (1.0 + drho)


def _dev(a, dtype=torch.int64):
    return torch.from_numpy(np.asarray(a).astype(np.int64 if dtype == torch.int64 else np.float64)).to("cuda", dtype)


class _Level:
    """One level's time step on pre-collision populations (27, N) in 64 bits."""

    def __init__(self, grid, omega, bounce_back=False):
        self.grid, self.omega = grid, float(np.float32(omega))
        self.fluid = None if grid.fluid.size == grid.N else torch.from_numpy(grid.geo == 19).cuda()
        self.lists = []
        for name in ("velocity", "noslip", "geometry"):
            bc = grid.bcs.get(name)
            if bc is not None and bc.n:
                q = np.asarray(bc.q27).reshape(27, bc.n).astype(np.float32)
                d, i = np.nonzero((q >= 0) & (q <= 1) & (np.arange(27) > 0)[:, None])
                wall = None if bc.velocity is None else torch.stack([_dev(np.float32(v), torch.float64) for v in bc.velocity])
                self.lists.append((name, _dev(bc.k), _dev(d), _dev(i), _dev(q[d, i], torch.float64), wall))
        self.bounce_back = bounce_back

    def _links(self, post, k, d, i, q, wall):
        """The populations that a list sends back along its links."""
        c, w = (torch.tensor(t, dtype=post.dtype, device=post.device) for t in (C, W))
        r = torch.tensor(OPPOSITE, device=post.device)[d]
        at = post[:, k]
        out, back = at[d, i], at[r, i]
        lid = 0.0 if wall is None else 6 * w[d] * (c[d] * wall[:, i].T).sum(1)
        if self.bounce_back:
            return r, k[i], out - lid
        drho, u = _flow_moments(at)
        drho, u = drho[i], u[:, i]
        cu = (c[d] * u.T).sum(1)
        feq = w[d] * (drho + (1 + drho) * (4.5 * cu * cu - 1.5 * (u * u).sum(0)))
        om = self.omega
        v = (1 - q) / (1 + q) * 0.5 * (out - back + (out + back - 2 * feq * om) / (1 - om))
        return r, k[i], v + (q * (out + back) - lid) / (1 + q)

    def step(self, pre, phi=None, inflow=None):
        if torch.is_grad_enabled():
            post = _collide(pre, self.omega, phi)
        else:
            post, chunk = torch.empty_like(pre), 1 << 21
            for a in range(0, pre.shape[1], chunk):
                part = None if phi is None else phi[a:a + chunk]
                post[:, a:a + chunk] = _collide(pre[:, a:a + chunk].contiguous(), self.omega, part)
        if self.fluid is not None:
            post = torch.where(self.fluid, post, pre[OPPOSITE])
        new = _streamed(post, self.grid)
        for name, k, d, i, q, wall in self.lists:
            r, node, v = self._links(post, k, d, i, q, inflow if name == "velocity" and inflow is not None else wall)
            new = new.index_put((r, node), v)
        bc = self.grid.bcs.get("pressure")
        if bc is not None and bc.n:
            near = new[:, _dev(bc.kN)]
            drho, u = _flow_moments(near)
            target = _dev(np.float32(bc.rho_bc), torch.float64)
            c, w = (torch.tensor(t, dtype=new.dtype, device=new.device) for t in (C, W))
            cu = c @ u
            shape = 1 + 3 * cu + 4.5 * cu * cu - 1.5 * (u * u).sum(0)
            v = near + w[:, None] * (target - drho) * shape
            axis, sign = (bc.direction - 1) // 2, 1 if bc.direction % 2 else -1
            rows = torch.tensor([j for j in range(27) if C[j][axis] * sign <= 0], device=new.device)
            new = new.index_put((rows[:, None], _dev(bc.k)[None, :]), v[rows])
        return new


_CORNERS = [(x, y, z) for z in (0, 1) for y in (0, 1) for x in (0, 1)]


def _corner_nodes(grid, base):
    x, y, z = (np.asarray(a)[np.asarray(base, dtype=np.int64)] for a in _coords(grid.nx, grid.ny, grid.nz))
    return torch.stack([_dev((x + a) % grid.nx + grid.nx * ((y + b) % grid.ny + grid.ny * ((z + c) % grid.nz)))
                        for a, b, c in _CORNERS])


@functools.lru_cache(maxsize=4)
def _coords(nx, ny, nz):
    k = np.arange(nx * ny * nz)
    return k % nx, k // nx % ny, k // (nx * ny)


def _polynomials(pre, corners, omega):
    """The compact second-order interpolation of velocity (from the corner values and the strain that
    the non-equilibrium moments give) and the trilinear density of every cell, as dicts of
    coefficients {(i, j, k): value} of x^i y^j z^k, corners at +-1/2."""
    f = pre[:, corners]  # (27, 8, cells)
    c = torch.tensor(C, dtype=f.dtype, device=f.device)
    drho = f.sum(0)
    rho = 1 + drho
    u = torch.einsum("da,dns->ans", c, f) / rho
    second = torch.einsum("da,db,dns->abns", c, c, f) / rho - u[:, None] * u[None]
    k = {(a, b): -3 * omega * second[a, b] for a, b in ((0, 1), (1, 2), (0, 2))}
    xy, xz = (-1.5 * omega * (second[0, 0] - second[a, a]) for a in (1, 2))
    sign = 2.0 * torch.tensor(_CORNERS, dtype=f.dtype, device=f.device) - 1.0  # (8, 3)

    def s(q, *axes):
        weight = torch.ones(8, dtype=f.dtype, device=f.device)
        for a in axes:
            weight = weight * sign[:, a]
        return weight @ q

    velocity = []
    # differences of the normal stresses seen from each axis: k_aa - k_bb for the two others
    diff = {(0, 1): xy, (0, 2): xz, (1, 0): -xy, (1, 2): xz - xy, (2, 0): -xz, (2, 1): xy - xz}
    for a in range(3):
        b, g = [i for i in range(3) if i != a]
        kab, kag = k[min(a, b), max(a, b)], k[min(a, g), max(a, g)]
        e = lambda **p: tuple(p.get("xyz"[i], 0) for i in range(3))  # noqa: E731
        name = "xyz"
        A = {}
        A[e()] = (8 * s(u[a]) + 2 * (s(u[b], a, b) + s(u[g], a, g) - s(kab, b) - s(kag, g))
                  - s(diff[a, b], a) - s(diff[a, g], a)) / 64
        A[e(**{name[a]: 2})] = (2 * (s(u[b], a, b) + s(u[g], a, g)) + s(diff[a, b], a) + s(diff[a, g], a)) / 16
        for o, ko in ((b, kab), (g, kag)):
            A[e(**{name[o]: 2})] = (s(ko, o) - 2 * s(u[o], a, o)) / 8
        for o in range(3):
            A[e(**{name[o]: 1})] = s(u[a], o) / 4
        for o, q in ((0, 1), (0, 2), (1, 2)):
            A[e(**{name[o]: 1, name[q]: 1})] = s(u[a], o, q) / 2
        A[1, 1, 1] = s(u[a], 0, 1, 2)
        velocity.append(A)
    density = {(0, 0, 0): s(drho) / 8, (1, 1, 1): s(drho, 0, 1, 2)}
    for o in range(3):
        density[tuple(int(i == o) for i in range(3))] = s(drho, o) / 4
    for o, q in ((0, 1), (0, 2), (1, 2)):
        density[tuple(int(i in (o, q)) for i in range(3))] = s(drho, o, q) / 2
    unit = [tuple(int(i == o) for i in range(3)) for o in range(3)]
    laplace = -3 * sum(velocity[a][unit[a]] ** 2 for a in range(3)) - 6 * sum(
        velocity[b][unit[a]] * velocity[a][unit[b]] for a, b in ((0, 1), (0, 2), (1, 2)))
    return velocity, density, laplace


def _value(poly, at):
    return sum(v * at[0] ** i * at[1] ** j * at[2] ** k for (i, j, k), v in poly.items())


def _slope(poly, axis, at):
    total = 0.0
    for p, v in poly.items():
        if p[axis]:
            q = [p[i] - (i == axis) for i in range(3)]
            total = total + v * p[axis] * at[0] ** q[0] * at[1] ** q[1] * at[2] ** q[2]
    return total


def _rebuilt(velocity, press, at, scale):
    """Populations of a node at `at` of the cell from the polynomials; scale: eps / omega."""
    u = torch.stack([_value(p, at) for p in velocity])
    g = [[_slope(velocity[a], b, at) for b in range(3)] for a in range(3)]
    k = scale * (1 + press)
    xy, xz = -2 / 3 * (g[0][0] - g[1][1]) * k, -2 / 3 * (g[0][0] - g[2][2]) * k
    m = {(i // 9, i // 3 % 3, i % 3): torch.zeros_like(press) for i in range(27)}
    m[0, 0, 0] = press
    m[2, 0, 0], m[0, 2, 0], m[0, 0, 2] = (xy + xz + press) / 3, (xz - 2 * xy + press) / 3, (xy - 2 * xz + press) / 3
    m[1, 1, 0], m[1, 0, 1], m[0, 1, 1] = (-1 / 3 * (g[a][b] + g[b][a]) * k for a, b in ((0, 1), (0, 2), (1, 2)))
    m[2, 2, 0] = m[2, 0, 2] = m[0, 2, 2] = press / 9
    m[2, 2, 2] = press / 27
    return _list(_from_central(_rest_moments(m), u))


class _Pair:
    """A coarse level and the refined box in it."""

    def __init__(self, case):
        nb = _nested(case["nx"], case["ny"], case["nz"])
        self.nb = nb
        self.coarse = _Level(nb.coarse, case["omega"])
        self.fine = _Level(nb.fine, _fine_omega(case["omega"]))
        self.fc = _corner_nodes(nb.fine, nb.fc.fine), _dev(nb.fc.coarse)
        self.cf = _corner_nodes(nb.coarse, nb.cf.coarse), _corner_nodes(nb.fine, nb.cf.fine)

    def step(self, pc, pf, phi, inflow):
        pf = self.fine.step(self.fine.step(pf, phi), phi)
        pc = self.coarse.step(pc, None, inflow)
        velocity, density, laplace = _polynomials(pf, self.fc[0], self.fine.omega)
        zero = (0.0, 0.0, 0.0)
        node = _rebuilt(velocity, _value(density, zero) - 0.25 * laplace, zero, 2.0 / self.coarse.omega)
        pc = pc.index_put((torch.arange(27, device="cuda")[:, None], self.fc[1][None, :]), node)
        velocity, density, laplace = _polynomials(pc, self.cf[0], self.coarse.omega)
        nodes = []
        for corner in _CORNERS:
            at = tuple(0.5 * v - 0.25 for v in corner)
            nodes.append(_rebuilt(velocity, _value(density, at) + 3 * at[0] ** 2 * laplace, at, 0.5 / self.fine.omega))
        nodes = torch.stack(nodes, 1)  # (27, 8, cells)
        pf = pf.index_put((torch.arange(27, device="cuda")[:, None, None], self.cf[1][None]), nodes)
        return pc, pf


def _drag_cells(grid):
    """The sphere's links: direction, node across, opposite direction, node, velocity."""
    bc = grid.bcs["geometry"]
    q = np.asarray(bc.q27).reshape(27, bc.n)
    d, i = np.nonzero((q >= 0) & (q <= 1) & (np.arange(27) > 0)[:, None])
    k = np.asarray(bc.k, dtype=np.int64)[i]
    x, y, z = (a[k] for a in _coords(grid.nx, grid.ny, grid.nz))
    c = np.array(C)[d]
    across = (x + c[:, 0]) % grid.nx + grid.nx * ((y + c[:, 1]) % grid.ny + grid.ny * ((z + c[:, 2]) % grid.nz))
    return _dev(d), _dev(across), _dev(np.array(OPPOSITE)[d]), _dev(k), _dev(c.T, torch.float64)


def _drag(pre, cells):
    d, across, r, k, c = cells
    return c @ (pre[d, across] + pre[r, k])


def exact(case, seed):
    kind = case["kind"]
    s = _inputs(case, seed)
    if kind == "two_level":
        with torch.no_grad():
            pair = _Pair(case)
            pc, pf = (_pre_of_buffer(f, g, True) for f, g in zip(s.f, (pair.nb.coarse, pair.nb.fine)))
            ux = (s.amplitudes @ s.basis).double()
            inflow = torch.stack([ux, torch.zeros_like(ux), torch.zeros_like(ux)])
            for _ in range(case["steps"]):
                pc, pf = pair.step(pc, pf, s.porosity.double(), inflow)
            return {"coarse": _buffer_of_pre(pc, pair.nb.coarse, case["steps"] % 2 == 0),
                    "fine": _buffer_of_pre(pf, pair.nb.fine, True)}
    if kind == "two_level_grad":
        pair = _Pair(case)
        pc, pf = (_pre_of_buffer(f, g, True) for f, g in zip(s.f, (pair.nb.coarse, pair.nb.fine)))
        a = s.amplitudes.double().requires_grad_(True)
        phi = s.porosity.double().requires_grad_(True)
        ux = a @ s.basis.double()
        inflow = torch.stack([ux, torch.zeros_like(ux), torch.zeros_like(ux)])
        nodes = _dev(_observed(pair.nb))
        J = 0.0
        for t in range(case["steps"]):
            pc, pf = checkpoint(pair.step, pc, pf, phi, inflow, use_reentrant=False)
            if t >= case["steps"] // 2:
                drho, u = _flow_moments(pc[:, nodes])
                J = J + (0.5 * (u * u).sum(0) * (1 + drho)).sum()
        ga, gp = torch.autograd.grad(J, (a, phi))
        return {"coarse": _buffer_of_pre(pc.detach(), pair.nb.coarse, case["steps"] % 2 == 0),
                "fine": _buffer_of_pre(pf.detach(), pair.nb.fine, True), "objective": J.detach(), "amplitude_grad": ga,
                "porosity_grad": gp}
    grid = _grid(case)
    level = _Level(grid, case["omega"], bounce_back=kind == "cavity")
    pre = _pre_of_buffer(s.f, grid, True)
    s.f = None
    phi = None if s.porosity is None else s.porosity.double()
    if kind == "sphere_grad":
        phi = phi.requires_grad_(True)
        cells = _drag_cells(grid)
        J = 0.0
        for t in range(case["steps"]):
            pre = checkpoint(level.step, pre, phi, use_reentrant=False)
            if t >= case["steps"] // 2:
                J = J + _drag(pre, cells)[0] / case["steps"]
        (gp,) = torch.autograd.grad(J, phi)
        return {"populations": _buffer_of_pre(pre.detach(), grid, case["steps"] % 2 == 0), "objective": J.detach(),
                "porosity_grad": gp}
    with torch.no_grad():
        if kind == "monitor":
            drho, u = _flow_moments(pre)
            energy = 0.5 * (u * u).sum(0) * (1 + drho)
            trace = (torch.tensor(C, dtype=pre.dtype, device=pre.device) ** 2).sum(1) @ pre
            press = 0.5 * (trace - drho - (u * u).sum(0) * (1 + drho)) + drho
            return {"sums": torch.stack([drho.sum(), *(u * (1 + drho)).sum(1), energy.sum()]).cpu().numpy(),
                    "energy": float(energy.sum()), "nodes": None, "rho": drho, "vx": u[0], "vy": u[1], "vz": u[2],
                    "pressure": press}
        drag = []
        cells = _drag_cells(grid) if kind == "sphere" else None
        for t in range(case["steps"] * case.get("rounds", 1)):
            pre = level.step(pre, phi)
            if cells is not None and (t + 1) % case["steps"] == 0:
                drag.append(_drag(pre, cells).cpu().numpy())
        buf = _buffer_of_pre(pre, grid, case["steps"] * case.get("rounds", 1) % 2 == 0)
        return {"populations": buf, "drag": np.stack(drag)} if cells is not None else {"populations": buf}
