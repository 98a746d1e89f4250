"""Which kernel the dense-box collision takes for a row of the FP16 types, seen from its roundings: the
row kernel and the one-node-per-thread kernel round FP16 differently, so a change of the choice changes
results. A working set beyond the cache is declared, not allocated."""
import ctypes

import numpy as np
import pytest

from helpers import near_equilibrium, pack_pre
from virtualfluids_amd.grid import periodic_box

pytestmark = pytest.mark.gpu


# rows of up to four whole waves at two or four nodes a lane (128, 256, 384, 512, 768, 1024 nodes) are the
# row kernel's, longer ones and those of five and seven waves at two (640, 896) the other's
@pytest.mark.parametrize("nx,row", [(128, True), (256, True), (384, True), (512, True), (768, True), (1024, True),
                                    (640, False), (896, False), (1280, False), (1536, False), (2048, False)])
def test_fp16_rows_keep_their_kernel(gpu, nx, row):
    import torch

    from virtualfluids_amd import capi
    from virtualfluids_amd.lattice import Lattice, stream_handle

    g = periodic_box(nx, 9, 7)
    pre = near_equilibrium(np.random.default_rng(nx), g.N, u_amp=0.04, noise=5e-3)
    out = {}
    for name, kernel in (("auto", capi.BOX_KERNEL_AUTO), ("row", capi.BOX_KERNEL_ROW), ("node", capi.BOX_KERNEL_NODE)):
        L = Lattice(g, 1.7, storage="fp16")
        L.set_working_set(1 << 32)
        L.param.kernelChoice.boxKernel = kernel
        L.set_populations(pack_pre(pre, g, True))
        into = torch.zeros_like(L.f)
        capi.call("vf_k17_run_box_into", L.pref(), ctypes.c_void_p(into.data_ptr()), stream_handle())
        L.collide()
        out[name] = (L.f.clone(), into)
    for i in range(2):
        assert torch.equal(out["auto"][i], out["row" if row else "node"][i])
        if row:
            assert not torch.equal(out["row"][i], out["node"][i])
