"""Macroscopic fields, moment sums and kinetic energy of boxes whose planes are thin or many (nodes
numbered flat, their coordinates by multiplication) against the neighbour-array forms of the same lattice."""
import numpy as np
import pytest

from helpers import near_equilibrium, pack_pre
from virtualfluids_amd.grid import GEO_SOLID, periodic_box

pytestmark = pytest.mark.gpu


def _results(g, pre, storage, even, box, addressing=0):
    from virtualfluids_amd.lattice import Lattice

    L = Lattice(g, 1.7, storage=storage, box=box)
    L.param.kernelChoice.rowAddressing = addressing
    L.set_populations(pack_pre(pre, g, even))
    L.even = even
    return [a.copy() for a in L.macroscopic()], np.asarray(L.moment_sums()), L.kinetic_energy()


# more planes than a launch has in y (65535), planes of four nodes, rows and columns only; either side
# of the 49152 nodes where the sums take larger workgroups
@pytest.mark.parametrize("shape", [(1, 1, 70000), (2, 2, 9000), (70000, 1, 1), (1, 49153, 1), (3, 1, 16384)])
@pytest.mark.parametrize("storage", ["fp32", "fp16"])
@pytest.mark.parametrize("solid", [False, True])
def test_thin_boxes(gpu, shape, storage, solid):
    g = periodic_box(*shape)
    rng = np.random.default_rng(3)
    if solid:
        s = rng.random(g.N) < 0.1
        g.geo = np.where(s, GEO_SOLID, g.geo).astype(np.uint32)
        g.fluid = np.nonzero(~s)[0].astype(np.uint32)
    pre = near_equilibrium(rng, g.N, noise=5e-3)
    for even in (True, False):
        (fa, sa, ea), (fb, sb, eb) = (_results(g, pre, storage, even, box) for box in (True, False))
        for a, b in zip(fa, fb):
            np.testing.assert_allclose(a, b, rtol=0, atol=2e-7)
            assert not solid or not np.any(a[s])
        np.testing.assert_allclose(sa, sb, rtol=1e-12, atol=1e-12 * g.N)
        assert ea[1] == eb[1]
        np.testing.assert_allclose(ea[0], eb[0], rtol=1e-6)
