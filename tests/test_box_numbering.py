"""The division by a box's plane and row in the kernels that number its nodes flat (vf_lattice.h, Divider):
k / d as (4 k m >> 32) >> s with m = floor(2^(30+s) / d) + 1, exact for every k < 2^30. The worst cases
are the ends of rows, near 2^30 above all."""
import numpy as np


def _divider(d):
    s = (d - 1).bit_length()
    return (1 << (30 + s)) // d + 1, s


def test_division_is_exact_at_the_ends_of_rows():
    rng = np.random.default_rng(2)
    top = 1 << 30
    for d in [*range(1, 2049), *rng.integers(2049, 1 << 20, 3000), *rng.integers(1 << 20, top, 500), top - 1,
              *(1 << b for b in range(30)), *((1 << b) + 1 for b in range(1, 29)), *((1 << b) - 1 for b in range(2, 31))]:
        d = int(d)
        m, s = _divider(d)
        assert m < 1 << 32
        rows = np.unique(np.concatenate([np.arange(64), rng.integers(0, top // d + 1, 64), [top // d - 1, top // d]]))
        for r in (0, d - 1):
            k = rows * d + r
            k = k[(k >= 0) & (k < top)].astype(np.uint64)
            q = ((k * np.uint64(4) * np.uint64(m)) >> np.uint64(32)) >> np.uint64(s)
            assert np.array_equal(q, k // np.uint64(d)), (d, r)
