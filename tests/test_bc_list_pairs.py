"""When a velocity and a no-slip list may share a launch (bc_post_pair_kernel): judged on the values
that the kernels see, at a cost that follows the lists."""
from types import SimpleNamespace

import numpy as np
import pytest

from virtualfluids_amd.grid import CX, CY, CZ
from virtualfluids_amd.simulation import _independent


def _grid(size, lists):
    nx, ny, nz = size
    return SimpleNamespace(nx=nx, ny=ny, nz=nz, N=nx * ny * nz, bcs=lists)


def _list(k, links):
    """Nodes k; links: [(direction, entry, distance)]."""
    q = np.full((27, len(k)), -1.0)
    for d, i, value in links:
        q[d, i] = value
    return SimpleNamespace(k=np.asarray(k, dtype=np.int32), n=len(k), q27=q.ravel())


# the kernels read FP32: 1 + 1e-9 rounds to 1 and -1e-60 to -0, links both; 1 + 1e-6 and -1e-30 stay outside
@pytest.mark.parametrize("q,link", [(1.0, True), (1.0 + 1e-9, True), (-1e-60, True), (1.0 + 1e-6, False),
                                    (-1e-30, False), (float("nan"), False), (-1.0, False)])
@pytest.mark.parametrize("swap", [False, True])
def test_links_are_those_of_the_fp32_distances(q, link, swap):
    size = (8, 8, 8)
    at = 3 + 8 * (3 + 8 * 3)
    for d in (1, 7, 26):
        to = at + CX[d] + 8 * (CY[d] + 8 * CZ[d])
        lists = [_list([at], [(d, 0, q)]), _list([to, 0], [])]
        if swap:
            lists.reverse()
        assert _independent(_grid(size, {"a": lists[0], "b": lists[1]}), "a", "b") == (not link)
        shared = [_list([at], [(d, 0, q)]), _list([at], [(d, 0, 0.5)])]
        if swap:
            shared.reverse()
        assert _independent(_grid(size, {"a": shared[0], "b": shared[1]}), "a", "b") == (not link)


def test_memory_follows_the_lists():
    """A few nodes in opposite corners of a box of 10^9 nodes: nothing of the box's size is held."""
    import resource

    size = (1000, 1000, 1000)
    N = 10 ** 9
    a, b = _list([0, N - 1], [(1, 0, 0.5)]), _list([5, N // 2, N - 7], [(2, 1, 0.5)])
    before = resource.getrusage(resource.RUSAGE_SELF).ru_maxrss
    assert _independent(_grid(size, {"a": a, "b": b}), "a", "b")
    assert resource.getrusage(resource.RUSAGE_SELF).ru_maxrss - before < 64 * 1024  # KiB
    b.k[0] = 1  # where a's first node has its link
    assert not _independent(_grid(size, {"a": a, "b": b}), "a", "b")


def test_no_memory_for_the_search_keeps_the_launches(tmp_path):
    """Without memory for the search the lists count as dependent: two launches, and no error that a
    run of steps would raise. In a process of its own, whose address space ends before the search's."""
    import subprocess
    import sys

    code = """
import ctypes, resource
import numpy as np
from virtualfluids_amd import capi
lib = capi.load()
n = 6_000_000
k = np.arange(n, dtype=np.int32)
q = np.zeros(27, dtype=np.float64)  # read for nodes beside the other list only: none here
far = k + np.int32(450 * 900 ** 2)
out = ctypes.c_int32(7)
p = lambda a: a.ctypes.data_as(ctypes.c_void_p)
used = int(open("/proc/self/statm").read().split()[0]) * resource.getpagesize()
resource.setrlimit(resource.RLIMIT_AS, (used + (16 << 20), resource.RLIM_INFINITY))
rc = lib.vf_bc_lists_independent(900, 900, 900, n, p(k), p(q), n, p(far), p(q), ctypes.byref(out))
print(rc, out.value)
"""
    r = subprocess.run([sys.executable, "-c", code], capture_output=True, text=True, timeout=120)
    assert r.stdout.split() == ["0", "0"], (r.stdout, r.stderr)


def _channel():
    from virtualfluids_amd.grid import sphere_channel
    from virtualfluids_amd.lattice import Lattice
    from virtualfluids_amd.simulation import BoundaryConditionFactory as F, Simulation

    f = F()
    f.set_velocity_boundary_condition(F.VelocityBC.VelocityInterpolatedCompressible)
    f.set_no_slip_boundary_condition(F.NoSlipBC.NoSlipInterpolatedCompressible)
    f.set_geometry_boundary_condition(F.NoSlipBC.NoSlipInterpolatedCompressible)
    f.set_pressure_boundary_condition(F.PressureBC.PressureNonEquilibriumCompressible)
    L = Lattice(sphere_channel((16, 10, 10), (6, 5, 5), 2.4, 0.04), 1.7, device="cpu")
    return Simulation(L, f)


def _shared_link(velocity, walls):
    """(direction, entry of the walls) of a node in both lists, along a link of the velocity list."""
    kv, kw = velocity.k.numpy(), walls.k.numpy()
    node = np.intersect1d(kv, kw)[0]
    qv = velocity.q27.numpy().reshape(27, -1)[:, np.flatnonzero(kv == node)[0]]
    return next(d for d in range(1, 27) if 0 <= qv[d] <= 1), int(np.flatnonzero(kw == node)[0])


@pytest.mark.parametrize("change", ["q27", "k", "pointer", "before"])
def test_lists_changed_on_the_device_are_judged_as_they_are(change):
    """The launch reads the device lists: what they hold decides, and a pair whose lists changed since
    goes back to two launches (also where the lists would pass again)."""
    sim = _channel()
    if change == "before":
        groups = sim._post_groups()
    else:
        assert [len(bcs) for _, bcs in sim._post_launches(10 ** 6)] == [2]
        assert [len(bcs) for _, bcs in sim._post_launches(1)] == [2]
        groups = sim.groups
    (_, _, velocity), (_, _, walls) = groups
    d, i = _shared_link(velocity, walls)
    if change in ("q27", "before"):
        walls.q27.view(27, -1)[d, i] = 0.5
    elif change == "k":
        walls.k.copy_(walls.k.flip(0))
    else:
        walls.kept = walls.q27.clone()
        walls.struct.q27 = walls.kept.data_ptr()
    assert [len(bcs) for _, bcs in sim._post_launches(1)] == [1, 1]
    if change in ("q27", "before"):
        assert [len(bcs) for _, bcs in sim._post_launches(10 ** 6)] == [1, 1]


def test_a_given_stream_is_not_waited_for():
    """Judging reads the lists back, which waits for the current stream's work: not in a call whose
    caller asked for another one."""
    sim = _channel()
    assert [len(bcs) for _, bcs in sim._post_launches(10 ** 6, stream=object())] == [1, 1]
    assert [len(bcs) for _, bcs in sim._post_launches(1)] == [2]


def test_asking_waits_for_the_steps_that_pay_for_it(monkeypatch):
    """2 to 5 ns a node against 2 us a step: long lists ask later than the 512 steps of short ones."""
    from virtualfluids_amd import simulation

    asked = []
    monkeypatch.setattr(simulation, "paired_launches",
                        lambda lattice, groups: asked.append(1) or [(fn, [(name, bc)]) for name, fn, bc in groups])
    for nodes, steps in ((100, 512), (200_000, 512), (1_000_000, 2500)):
        sim = _channel()
        for _, _, bc in sim._post_groups():
            bc.n = nodes // 2
        asked.clear()
        sim._post_launches(steps - 1)
        assert not asked
        sim._post_launches(1)
        assert asked
