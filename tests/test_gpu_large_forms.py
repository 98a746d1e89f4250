"""The kernel forms of large lattices: 64-bit addresses pinned on small ones (against the oracle, against
the buffer descriptors), and lattices whose 14 slots reach beyond 4 GiB as they come."""
import ctypes

import numpy as np
import pytest

from helpers import near_equilibrium, pack_pre
from virtualfluids_amd import capi
from virtualfluids_amd.grid import CX, CY, CZ, periodic_box

pytestmark = pytest.mark.gpu


def _global(L):
    L.param.kernelChoice.rowAddressing = capi.ROW_ADDRESSING_GLOBAL
    return L


# the one-node-per-thread kernel of boxes and the kernel of neighbour arrays; tolerances of the oracle
# tests of the other forms: a few ulp, and one storage rounding of |f| < 0.06
@pytest.mark.parametrize("box", [True, False])
@pytest.mark.parametrize("storage,tol", [("fp32", 2e-7), ("fp16", 0.06 * 2.0 ** -11 + 2e-7),
                                         ("bf16", 0.06 * 2.0 ** -8 + 2e-7)])
@pytest.mark.parametrize("dims", [(64, 5, 3), (130, 4, 3)])
def test_64_bit_addresses_match_oracle(gpu, orc, box, storage, tol, dims):
    from virtualfluids_amd.lattice import Lattice

    g = periodic_box(*dims)
    f0 = near_equilibrium(np.random.default_rng(sum(dims)), g.N, u_amp=0.04, noise=5e-3)
    for even in (True, False):
        L = _global(Lattice(g, 1.9, storage=storage, box=box))
        L.param.kernelChoice.boxKernel = capi.BOX_KERNEL_NODE
        L.even = even
        L.set_populations(pack_pre(f0, g, even))
        ref = orc.Lattice(g.nbx, g.nby, g.nbz)
        ref.even = even
        ref.f[:] = L.populations().astype(np.float64)
        ref.collide(g.fluid, 1.9)
        L.collide()
        assert np.abs(L.populations() - ref.f).max() < tol


@pytest.mark.parametrize("storage", ["fp32", "fp16", "bf16"])
@pytest.mark.parametrize("shape", [(33, 31, 5), (64, 40, 20)])
def test_fields_and_sums_through_64_bit_addresses(gpu, storage, shape):
    from virtualfluids_amd.lattice import Lattice

    g = periodic_box(*shape)
    pre = near_equilibrium(np.random.default_rng(5), g.N, noise=5e-3)
    for even in (True, False):
        out = []
        for pinned in (False, True):
            L = Lattice(g, 1.7, storage=storage)
            if pinned:
                _global(L)
            L.set_populations(pack_pre(pre, g, even))
            L.even = even
            out.append(([a.copy() for a in L.macroscopic()], L.moment_sums()))
        for a, b in zip(out[0][0], out[1][0]):
            np.testing.assert_allclose(a, b, rtol=0, atol=2e-7)
        np.testing.assert_allclose(out[0][1], out[1][1], rtol=1e-12, atol=1e-12 * g.N)


# 83.5 M nodes (14 FP32 slots span 4.7 GB, 7 span 2.3) and 151 M (7 span 4.23 of 4.29 GB); rows of 448 and 512
@pytest.mark.parametrize("shape", [(448, 448, 416), (512, 512, 576)])
def test_lattices_beyond_two_descriptors(gpu, shape):
    import torch

    from virtualfluids_amd.lattice import stream_handle

    nx, ny, nz = shape
    N = nx * ny * nz
    gen = torch.Generator(device="cuda").manual_seed(nx)
    f0 = torch.empty(27 * N, dtype=torch.float32, device="cuda")
    for d in range(27):
        f0[d * N:(d + 1) * N].normal_(0.0, 1e-3, generator=gen)
    fields = torch.zeros((5, N), dtype=torch.float32, device="cuda")
    f = f0.clone()
    p = capi.LBMParameter()
    p.distributions, p.storage, p.isEvenTimestep, p.numberOfNodes = f.data_ptr(), capi.VF_STORAGE_FP32, 1, N
    p.nx, p.ny, p.nz, p.omega, p.forceFactor = nx, ny, nz, 1.7, 1.0
    p.quadricLimiters[:] = [0.01] * 3
    p.rho, p.velocityX, p.velocityY, p.velocityZ, p.pressure = (fields[i].data_ptr() for i in range(5))
    P, s = ctypes.byref(p), stream_handle()

    def slots_equal(a, b):
        return all(torch.equal(a[d * N:(d + 1) * N], b[d * N:(d + 1) * N]) for d in range(27))

    # the sums against torch's in 64 bits, the fields against their definition at nodes all over the box
    sums = torch.zeros(5, dtype=torch.float64, device="cuda")
    capi.call("vf_MomentSums", P, sums.data_ptr(), s)
    capi.call("vf_CalculateMacroscopicQuantitiesCompressible", P, s)
    per = torch.stack([f0[d * N:(d + 1) * N].double().sum() for d in range(27)]).cpu().numpy()
    want = [per.sum(), (CX * per).sum(), (CY * per).sum(), (CZ * per).sum()]
    # sums of 27 N terms of 1e-3, each rounded in 64 bits and added in another order
    np.testing.assert_allclose(sums[:4].cpu().numpy(), want, rtol=0, atol=27 * N * 1e-3 * 2.0 ** -52 * 64)
    k = torch.cat([torch.arange(64, device="cuda"), N - 1 - torch.arange(64, device="cuda"),
                   torch.randint(0, N, (4096,), device="cuda", generator=gen)])
    x, y, z = k % nx, k // nx % ny, k // (nx * ny)
    drho = torch.zeros(k.numel(), dtype=torch.float64, device="cuda")
    jx = torch.zeros_like(drho)
    for d in range(27):
        n = (x + int(CX[d] < 0)) % nx + nx * ((y + int(CY[d] < 0)) % ny + ny * ((z + int(CZ[d] < 0)) % nz))
        v = f0[d * N + n].double()
        drho += v
        jx += int(CX[d]) * v
    # 27 FP32 additions of terms of a few 1e-3
    assert float((fields[0][k].double() - drho).abs().max()) < 27 * 2e-2 * 2.0 ** -24
    assert float((fields[1][k].double() - jx / (1.0 + drho)).abs().max()) < 30 * 2e-2 * 2.0 ** -24

    # the automatic form (four descriptors) against 64-bit addresses: in place and out of place
    capi.call("vf_k17_run_box", P, capi.COLLISION_DEFAULT, s)
    stepped = f.clone()
    f.copy_(f0)
    p.kernelChoice.rowAddressing = capi.ROW_ADDRESSING_GLOBAL
    capi.call("vf_k17_run_box", P, capi.COLLISION_DEFAULT, s)
    assert slots_equal(f, stepped) and not torch.equal(f[:N], f0[:N])
    f.copy_(f0)
    del f0
    p.kernelChoice.rowAddressing = capi.ROW_ADDRESSING_AUTO
    into = torch.zeros_like(f)
    capi.call("vf_k17_run_box_into", P, into.data_ptr(), s)
    assert slots_equal(into, stepped)


@pytest.mark.parametrize("storage", ["fp32", "fp16", "bf16"])
@pytest.mark.parametrize("solid", [False, True])
def test_write_macro_vars_leaves_the_same_populations(gpu, storage, solid):
    """A collision that also writes the macroscopic values (64-bit addresses on 16-bit lattices that fit
    the cache) leaves the populations of the plain one."""
    import torch

    from virtualfluids_amd.grid import GEO_SOLID
    from virtualfluids_amd.lattice import Lattice

    g = periodic_box(33, 31, 6)
    rng = np.random.default_rng(9)
    if solid:
        s = rng.random(g.N) < 0.1
        g.geo = np.where(s, GEO_SOLID, g.geo).astype(np.uint32)
        g.fluid = np.nonzero(~s)[0].astype(np.uint32)
    pre = near_equilibrium(rng, g.N, u_amp=0.04, noise=5e-3)
    for even in (True, False):
        out = []
        for macro in (True, False):
            L = Lattice(g, 1.9, storage=storage)
            L.even = even
            L.set_populations(pack_pre(pre, g, even))
            L.collide(write_macro=macro)
            out.append(L.f.clone())
        assert torch.equal(*out)
