"""The out-of-place step of the one-node-per-thread kernel leaves what the in-place step leaves, solid nodes
included, bit for bit: small FP32 lattices store both kinds of node together, others apart."""
import ctypes

import numpy as np
import pytest

from helpers import near_equilibrium, pack_pre
from virtualfluids_amd.grid import GEO_SOLID, periodic_box

pytestmark = pytest.mark.gpu


# a workgroup part full; planes that end inside one; XCD ranges; either side of the 48 MiB line (FP32)
@pytest.mark.parametrize("shape", [(5, 7, 3), (33, 31, 6), (64, 20, 5), (66, 80, 80), (80, 80, 80)])
@pytest.mark.parametrize("storage", ["fp32", "fp16", "bf16"])
def test_out_of_place_equals_in_place(gpu, shape, storage):
    import torch

    from virtualfluids_amd import capi
    from virtualfluids_amd.lattice import Lattice, stream_handle

    g = periodic_box(*shape)
    rng = np.random.default_rng(g.N)
    solid = rng.random(g.N) < 0.1
    g.geo = np.where(solid, GEO_SOLID, g.geo).astype(np.uint32)
    g.fluid = np.nonzero(~solid)[0].astype(np.uint32)
    pre = near_equilibrium(rng, g.N, u_amp=0.04, noise=5e-3)
    porosity = rng.uniform(0.0, 0.05, g.N)
    for even in (True, False):
        L = Lattice(g, 1.9, storage=storage)
        L.param.kernelChoice.boxKernel = capi.BOX_KERNEL_NODE
        L.set_porosity(porosity if even else None)
        L.even = even
        L.set_populations(pack_pre(pre, g, even))
        before = L.f.clone()
        into = torch.zeros_like(L.f)
        capi.call("vf_k17_run_box_into", L.pref(), ctypes.c_void_p(into.data_ptr()), stream_handle())
        assert torch.equal(L.f, before)
        L.collide()
        assert torch.equal(into, L.f) and not torch.equal(into, before)
