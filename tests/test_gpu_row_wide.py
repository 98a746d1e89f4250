"""The row kernel through four buffer descriptors (lattices whose 14 slots reach beyond 4 GiB) and in
workgroups of up to 512 lanes: the same populations bit for bit as through two descriptors, in
place and out of place, with whole and partial rows, both parities and solid nodes."""
import numpy as np
import pytest

from helpers import near_equilibrium, pack_pre
from virtualfluids_amd.grid import GEO_SOLID, periodic_box

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dims", [(64, 5, 3), (258, 3, 3), (450, 2, 3), (512, 3, 2)])
@pytest.mark.parametrize("storage,width", [("fp32", 1), ("fp32", 2), ("fp16", 2), ("bf16", 2)])
@pytest.mark.parametrize("solid", [False, True])
def test_wide_descriptors_match_two(gpu, dims, storage, width, solid):
    import ctypes

    import torch

    from virtualfluids_amd import capi
    from virtualfluids_amd.lattice import Lattice, stream_handle

    g = periodic_box(*dims)
    rng = np.random.default_rng(23)
    if solid:
        s = rng.random(g.N) < 0.05
        g.geo = np.where(s, GEO_SOLID, g.geo).astype(np.uint32)
        g.fluid = np.nonzero(~s)[0].astype(np.uint32)
    pre = near_equilibrium(rng, g.N, u_amp=0.04, noise=5e-3)
    for even in (True, False):
        out = []
        for addressing in (capi.ROW_ADDRESSING_BUFFER, capi.ROW_ADDRESSING_BUFFER_WIDE, capi.ROW_ADDRESSING_GLOBAL):
            L = Lattice(g, 1.9, storage=storage)
            c = L.param.kernelChoice
            c.boxKernel, c.rowWidth, c.rowAddressing = capi.BOX_KERNEL_ROW, width, addressing
            L.even = even
            L.set_populations(pack_pre(pre, g, even))
            into = torch.zeros_like(L.f)
            capi.call("vf_k17_run_box_into", L.pref(), ctypes.c_void_p(into.data_ptr()), stream_handle())
            L.collide()
            out.append((L.f.clone(), into))
        for f, into in out:
            assert torch.equal(f, out[0][0]) and torch.equal(into, out[0][0])
