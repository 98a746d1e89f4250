"""A velocity list and a no-slip list in one launch (bc_post_pair_kernel) against the two launches:
the same populations, bit for bit; and the lists that must not share one."""
import numpy as np
import pytest

from virtualfluids_amd.grid import CX, CY, CZ, sphere_channel

NOSLIP, VELOCITY = "vf_NoSlipInterpolatedCompressible", "vf_VelocityInterpolatedCompressible"
PAIR = "vf_VelocityAndNoSlipInterpolatedCompressible"


def test_lists_that_touch_each_other_keep_their_launches():
    from types import SimpleNamespace

    from virtualfluids_amd.simulation import paired_launches

    def launches(grid, box=True):
        L = SimpleNamespace(grid=grid, box=box)
        return [fn for fn, _ in paired_launches(L, [("velocity", VELOCITY, None), ("noslip+geometry", NOSLIP, None)])]

    def channel():
        return sphere_channel((16, 10, 10), (6, 5, 5), 2.4, 0.04)

    assert launches(channel()) == [PAIR]
    assert launches(channel(), box=False) == [VELOCITY, NOSLIP]
    g = channel()  # a link in common
    v, w = g.bcs["velocity"], g.bcs["noslip"]
    node = np.intersect1d(v.k, w.k)[0]
    qv, qw = v.q27.reshape(27, v.n), w.q27.reshape(27, w.n)
    d = next(d for d in range(1, 27) if 0 <= qv[d, v.k == node][0] <= 1)
    qw[d, w.k == node] = 0.5
    assert launches(g) == [VELOCITY, NOSLIP]
    g = channel()  # a link of the walls that leads to an inflow node
    v, w = g.bcs["velocity"], g.bcs["noslip"]
    qw = w.q27.reshape(27, w.n)
    for d in range(1, 27):
        to = w.k + CX[d] + g.nx * (CY[d] + g.ny * CZ[d])
        hit = np.nonzero(np.isin(to, v.k))[0]
        if hit.size:
            qw[d, hit[0]] = 0.5
            break
    assert hit.size and launches(g) == [VELOCITY, NOSLIP]


def test_independence_of_lists_matches_a_search_over_links():
    """Random lists on tiny periodic boxes: the restricted table search against all pairs."""
    from types import SimpleNamespace as NS

    from virtualfluids_amd.simulation import _independent

    rng = np.random.default_rng(0)
    seen = set()
    for _ in range(400):
        nx, ny, nz = (int(n) for n in rng.integers(2, 7, 3))
        N = nx * ny * nz

        def index(x, y, z):
            return x + nx * (y + ny * z)

        def random_list():
            k = rng.choice(N, min(int(rng.integers(1, 4)), N), replace=False).astype(np.int32)
            q = np.where(rng.random((27, k.size)) < 0.12, rng.random((27, k.size)), -1.0)
            return NS(k=k, n=k.size, q27=q.ravel())

        bcs = {name: random_list() for name in "abc"}
        expected = True
        for A, B in [(bcs["a"], bcs["b"]), (bcs["a"], bcs["c"])]:
            for H, O in ((A, B), (B, A)):
                for i, k in enumerate(H.k):
                    for d in range(1, 27):
                        if H.q27[d * H.n + i] < 0:
                            continue
                        x, y, z = k % nx, k // nx % ny, k // (nx * ny)
                        to = index((x + CX[d]) % nx, (y + CY[d]) % ny, (z + CZ[d]) % nz)
                        shared = any(j == k and O.q27[d * O.n + m] >= 0 for m, j in enumerate(O.k))
                        expected &= to not in O.k and not shared
        grid = NS(nx=nx, ny=ny, nz=nz, N=N, index=index, bcs=bcs)
        assert _independent(grid, "a", "b+c") == expected
        seen.add(expected)
    assert seen == {True, False}


# thread and lane forms; lists that end inside a workgroup (inflow of 6 x 5 nodes: 15 lane
# workgroups) and of many workgroups
@pytest.mark.gpu
@pytest.mark.parametrize("storage", ["fp32", "fp16", "bf16"])
@pytest.mark.parametrize("size", [(9, 6, 5), (40, 21, 18)])
@pytest.mark.parametrize("rows", [None, (0, 0), (1, 0), (0, 1), (1, 1)])
@pytest.mark.parametrize("velocity_bc", ["VelocityInterpolatedCompressible",
                                         "VelocityWithPressureInterpolatedCompressible"])
def test_pair_matches_two_launches(gpu, storage, size, rows, velocity_bc):
    import torch

    from virtualfluids_amd.lattice import Lattice
    from virtualfluids_amd.simulation import BoundaryConditionFactory as F, Simulation

    nx, ny, nz = size
    grid = sphere_channel(size, (nx // 3, ny // 2, nz // 2), min(ny, nz) / 4.0, 0.05, wall_q=0.3)
    rng = np.random.default_rng(nx)
    for bc in grid.bcs.values():  # a distance of its own for every active link, both ends included
        q = np.asarray(bc.q27)
        bc.q27 = np.where((q >= 0) & (q <= 1), rng.choice([0.0, 1.0, 0.5, 0.137, 0.81], q.size), q)
    init = [0.02 * rng.standard_normal(grid.N) for _ in range(4)]
    out = []
    for pair in (True, False):
        L = Lattice(grid, 1.7, storage=storage, box=True)
        L.init_equilibrium(*init)
        if rows is not None:
            for name, bc in L.bcs.items():
                bc.struct.nodesAlongRows = rows[0 if name == "velocity" else 1]
        f = F()
        f.set_velocity_boundary_condition(getattr(F.VelocityBC, velocity_bc))
        f.set_no_slip_boundary_condition(F.NoSlipBC.NoSlipInterpolatedCompressible)
        f.set_geometry_boundary_condition(F.NoSlipBC.NoSlipInterpolatedCompressible)
        f.set_pressure_boundary_condition(F.PressureBC.PressureNonEquilibriumCompressible)
        sim = Simulation(L, f)
        launches = sim._post_launches(512)
        assert len(launches[0][1]) == 2
        if not pair:
            sim._paired = (sim.groups, [(fn, [(name, bc)]) for name, fn, bc in sim.groups])
        sim.run(5)
        sim.step()
        torch.cuda.synchronize()
        out.append(L.f.clone())
    a, b = (t.view(torch.int32 if storage == "fp32" else torch.int16) for t in out)
    assert torch.isfinite(out[0].float()).all()
    assert int((a != b).sum()) == 0
