"""Sizes at the edges of the kernels' tiles and of their launch rules, against
the oracle (bit for bit where the kernels perform the reference's operations
in its order)."""
import numpy as np
import pytest

import cases
from oracle import Oracle

pytestmark = pytest.mark.gpu

eif = pytest.importorskip("ellipsesinflows_amd")


def potential(nx, ny, ly, mode=eif.POISSON_THOMAS):
    """psi of the same random velocities on the GPU and by the oracle"""
    kw = dict(itot=nx, jtot=ny, ly=ly, Re=100.0, extfrcy=0.1)
    g, o = eif.Solver(poisson_mode=mode, **kw), Oracle(**kw)
    ux, uy, p = cases.random_fields(nx, ny, nx * 7 + ny)
    for s in (g, o):
        s.upload(ux, uy, p)
        s.update_boundaries()
        s.set_dt(1e-3)
        s.compute_potential(1)
    out = g.field("psi"), o.field("psi")
    g.close()
    return out


# the sweep's tiles hold 128 rows of 16 wavenumbers and cover jtot - 1 rows:
# one row, one short of and one past one, two and three tiles, and
# wavenumber counts that leave a partial block; ly = 1e9 makes the first
# pivots vanish against the reference's absolute threshold (the zero-pivot
# form of the kernel)
@pytest.mark.parametrize("nx,ny,ly", [(16, 3, 1.0), (17, 4, 1.0), (64, 17, 1.0), (48, 128, 1.0),
                                      (33, 129, 1.0), (16, 130, 1.0), (64, 256, 2.0),
                                      (20, 257, 1.0), (31, 258, 1.0), (128, 385, 1.0),
                                      (64, 512, 2.0), (16, 12, 1e9), (16, 140, 1e9)])
def test_thomas_sweep_bit_exact_at_tile_edges(nx, ny, ly):
    a, b = potential(nx, ny, ly)
    assert np.array_equal(a, b)


# row lengths of every pass of the transform of any length: each register
# form alone and after others (12 = 2 2 3, 14 = 2 7, 20 = 2 2, 5, 30 = 2 3, 5,
# 90 = 2 3, 3 5, 98 = 2 7, 7, 147 = 3, 7, 7, 375 = 3 5, 5, 5,
# 768 = 2 2 2, 2 2 2, 2 2 3), radices summed over LDS first, last and
# repeated (11, 121, 22, 143, 499 prime), more groups than threads, and a row
# whose buffers exceed 64 KiB
@pytest.mark.parametrize("nx", [3, 9, 11, 12, 14, 20, 22, 30, 90, 98, 121, 143, 147, 375, 499,
                                768, 1701, 2500])
def test_transform_of_any_length_bit_exact(nx):
    a, b = potential(nx, 6, 0.5)
    assert np.array_equal(a, b)
