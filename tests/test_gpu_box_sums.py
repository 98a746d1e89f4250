"""The box forms of the macroscopic output, the FP64 moment sums and the kinetic energy (a workgroup
per piece of 1024 nodes of a plane) against the same sums in numpy and against the neighbour-array
forms of the same lattice: planes of one node less and more than a piece, more pieces than
workgroups, a single plane, and solid nodes."""
import numpy as np
import pytest

from helpers import near_equilibrium, pack_pre
from virtualfluids_amd.grid import CX, CY, CZ, GEO_SOLID, periodic_box

pytestmark = pytest.mark.gpu


# planes of 1023, 1024 and 1025 nodes; 1 x 1 x n; 2 pieces x 150 planes = 300 > 256 workgroups
@pytest.mark.parametrize("shape", [(33, 31, 5), (32, 32, 4), (41, 25, 3), (1, 1, 7), (40, 30, 150), (70, 90, 1)])
@pytest.mark.parametrize("storage", ["fp32", "fp16", "bf16"])
@pytest.mark.parametrize("even", [True, False])
def test_box_sums_and_fields(gpu, shape, storage, even):
    import torch

    from virtualfluids_amd.lattice import Lattice

    g = periodic_box(*shape)
    rng = np.random.default_rng(11)
    if g.N > 1000:
        solid = rng.random(g.N) < 0.03
        g.geo = np.where(solid, GEO_SOLID, g.geo).astype(np.uint32)
        g.fluid = np.nonzero(~solid)[0].astype(np.uint32)
    pre = near_equilibrium(rng, g.N, noise=5e-3)
    out = []
    for box in (True, False):
        L = Lattice(g, 1.7, storage=storage, box=box)
        L.set_populations(pack_pre(pre, g, even))
        L.even = even
        fields = [a.copy() for a in L.macroscopic()]
        out.append((fields, L.moment_sums(), L.kinetic_energy()))
    # the same node formulas: fields agree to FP32 round-off of the sums, the sums to FP64's
    for a, b in zip(out[0][0], out[1][0]):
        np.testing.assert_allclose(a, b, rtol=0, atol=2e-7)
    np.testing.assert_allclose(out[0][1], out[1][1], rtol=1e-12, atol=1e-12 * g.N)
    assert out[0][2][1] == out[1][2][1]
    np.testing.assert_allclose(out[0][2][0], out[1][2][0], rtol=1e-6)
    # and numpy's sums of the stored values over the fluid nodes
    dtype = {"fp32": torch.float32, "fp16": torch.float16, "bf16": torch.bfloat16}[storage]
    f = torch.from_numpy(np.ascontiguousarray(pre, dtype=np.float32)).to(dtype).double().numpy().T
    f = f[:, g.geo == 19]
    drho, j = f.sum(0), np.stack([c @ f for c in (CX, CY, CZ)])
    want = [drho.sum(), *j.sum(1), (0.5 * (j * j).sum(0) / (1.0 + drho)).sum()]
    np.testing.assert_allclose(out[0][1], want, rtol=1e-11, atol=1e-12 * g.N)
