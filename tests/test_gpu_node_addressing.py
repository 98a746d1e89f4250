"""The one-node-per-thread kernels (in place, out of place, bounce-back epilogue, adjoint) through
64-bit addresses, which boxes take whose 14 slots reach beyond 4 GiB, against the buffer
descriptors of smaller ones. The two forms differ by the compiler's contractions at most: a few
hundred FP32 roundings of terms below one (2e-6), and one step of a 16-bit storage type where such
a difference crosses a rounding boundary; the adjoint's terms reach the sum of 27 unit adjoints (1e-4)."""
import ctypes

import numpy as np
import pytest

from virtualfluids_amd.grid import cavity

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [5, 17])  # 7^3: less than a workgroup a plane; 19^3: planes end inside one
@pytest.mark.parametrize("storage,step", [("fp32", 0.0), ("fp16", 2.0 ** -10), ("bf16", 2.0 ** -7)])
def test_addresses_match_descriptors(gpu, n, storage, step):
    import torch

    from virtualfluids_amd import capi
    from virtualfluids_amd.lattice import Lattice, stream_handle
    from virtualfluids_amd.simulation import BoundaryConditionFactory as F, Simulation

    g = cavity(n)
    rng = np.random.default_rng(n)
    init = [0.02 * rng.standard_normal(g.N) for _ in range(4)]
    lam0 = torch.from_numpy(rng.standard_normal(27 * g.N).astype(np.float32)).cuda()
    f = F()
    f.set_velocity_boundary_condition(F.VelocityBC.VelocityBounceBack)
    f.set_no_slip_boundary_condition(F.NoSlipBC.NoSlipBounceBack)
    out = []
    for addressing in (capi.ROW_ADDRESSING_BUFFER, capi.ROW_ADDRESSING_GLOBAL):
        values = []
        for even in (True, False):
            L = Lattice(g, 1.7, storage=storage, box=True)
            c = L.param.kernelChoice
            c.boxKernel, c.rowAddressing, c.adjointKernel = (capi.BOX_KERNEL_NODE, addressing,
                                                             capi.ADJOINT_KERNEL_NODE)
            L.init_equilibrium(*init)
            L.even = even
            into, lam, start = torch.zeros_like(L.f), lam0.clone(), L.f.clone()
            capi.call("vf_k17_run_box_into", L.pref(), ctypes.c_void_p(into.data_ptr()), stream_handle())
            capi.call("vf_k17_adjoint_box", L.pref(), ctypes.c_void_p(lam.data_ptr()), None, None, stream_handle())
            sim = Simulation(L, f)
            assert sim.fused is not None
            sim.fused.run()
            fused = L.f.clone()
            L.f.copy_(start)
            L.collide()
            values += [into, fused, L.f.clone(), lam]
        torch.cuda.synchronize()
        out.append(values)
    for i, (a, b) in enumerate(zip(*out)):
        a, b = a.float(), b.float()
        assert torch.isfinite(a).all()
        if i % 4 == 3:
            assert float((a - b).abs().max()) <= 1e-4
        else:
            assert bool(((a - b).abs() <= 2e-6 + step * b.abs()).all())
