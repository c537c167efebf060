"""Sizes at the edges of the kernels' tiles and of their launch rules, against
the oracle (bit for bit where the kernels perform the reference's operations
in its order)."""
import concurrent.futures
import os

import numpy as np
import pytest
import torch

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


# bodies whose cells meet the foot search's special places: circles centred on
# a cell centre (every direction is a foot), thin ellipses (the evolute comes
# within a cell of the tip), tall ones, one across the periodic boundary, and
# a body smaller than a cell's diagonal; the sums of the weights' passes agree
# to the rounding of some 1e4 terms (1e-13 of the largest member)
@pytest.mark.parametrize("a,b,az", [(0.125, 0.125, 0.0), (0.2, 0.02, 0.0), (0.2, 0.02, 0.7),
                                    (0.02, 0.2, 1.1), (0.15, 0.149, 2.0), (0.012, 0.01, 0.3)])
def test_weights_of_special_shapes(a, b, az):
    nx = ny = 64
    kw = dict(itot=nx, jtot=ny, ly=1.0, Re=100.0)
    g, o = eif.Solver(**kw), Oracle(**kw)
    ux, uy, p = cases.random_fields(nx, ny, 5)
    parts = dict(den=[1.0, 1.2], a=[a, a], b=[b, b], x=[32.5 / nx, 0.37], y=[32.5 / ny, 0.99],
                 az=[az, az], ux=[0.3, -0.2], uy=[0.1, 0.4], vz=[0.5, -0.3])
    for s in (g, o):
        s.upload(ux, uy, p)
        s.update_boundaries()
        s.set_dt(1e-3)
        s.set_particles(**parts)
        s.reset_particle_increments()
        s.compute_inertia(0)
        s.exchange_momentum()
        # the warm starts, near and far: a small and a large increment
        rec = s.particles()
        rec[:, 6:9] = 1e-9
        s.set_particle_records(rec)
        s.compute_inertia(1)
        rec = s.particles()
        rec[:, 6:9] = [0.004, -0.003, 0.01]
        s.set_particle_records(rec)
        s.compute_inertia(1)
    x, y = g.particles(), o.particles()
    for cols in ((18, 19), (20, 21), (22, 23), (15, 16), (17,)):
        c = list(cols)
        assert np.max(np.abs(x[:, c] - y[:, c])) <= 1e-13 * max(np.max(np.abs(y[:, c])), 1.0), cols
    g.close()


# particle counts on either side of the wide workgroups of the increment, and
# partial workgroups
@pytest.mark.parametrize("n", [1, 5, 2047, 2048, 2065])
def test_increment_bit_exact_at_its_workgroup_sizes(n):
    kw = dict(itot=32, jtot=64, ly=2.0, Re=100.0, Fr=2.0)
    g, o = eif.Solver(**kw), Oracle(**kw)
    rng = np.random.default_rng(n)
    parts = dict(den=rng.uniform(1, 2, n), a=np.full(n, 0.003), b=np.full(n, 0.002),
                 x=rng.uniform(0.1, 0.9, n), y=rng.uniform(0, 2, n), az=rng.uniform(0, 3, n))
    for s in (g, o):
        s.set_dt(1e-2)
        s.set_particles(**parts)
        rec = s.particles()
        rec[:, 9:30] = np.random.default_rng(7).standard_normal((n, 21))
        s.set_particle_records(rec)
        res = s.increment_particles(1)
        s.res = res
    assert g.res == o.res
    assert np.array_equal(g.particles(), o.particles())
    g.close()


def objective(s, dts):
    """mean over the steps of the wall shear and the drag of the last exchange"""
    j = 0.0
    for dt in dts:
        s.step_fixed_dt(dt)
        rec = s.particles()
        j += s.wall_shear() - float(np.sum(rec[:, 0] * np.pi * rec[:, 1] * rec[:, 2] * rec[:, 16]))
    return j / len(dts)


# the gathered transposed stencils and the reversed weights on grids whose
# rows, columns and spacings are of every kind (two columns, odd, more columns
# than a workgroup), against central differences along a random direction of
# the velocity and of the particles: h = 1e-6 leaves h^2 J''' and round-off of
# about 1e-16 J / h = 1e-10 J, held here to 1e-7 of the derivative's scale
@pytest.mark.parametrize("nx,ny,ly", [(16, 12, 0.8), (33, 20, 1.0), (64, 31, 0.5), (270, 16, 0.06)])
def test_adjoint_along_a_direction(nx, ny, ly):
    kw = dict(itot=nx, jtot=ny, ly=ly, Re=40.0, extfrcy=0.2)
    rng = np.random.default_rng(nx)
    r = min(0.2 * ly, 0.15)
    parts = dict(den=[1.3], a=[r], b=[0.7 * r], x=[0.45], y=[0.02 * ly], az=[0.4], ux=[0.1],
                 uy=[-0.2], vz=[0.3])
    ux, uy, p = cases.random_fields(nx, ny, 11, amp=0.3)
    p[:] = 0.0
    dts = [2e-4, 2.5e-4]
    dux, duy = np.zeros_like(ux), np.zeros_like(uy)
    dux[1:-1, 1:-1] = rng.standard_normal((ny, nx - 1))
    duy[1:-1, 1:-1] = rng.standard_normal((ny, nx))
    dvel = rng.standard_normal(3)

    def solver(h):
        s = eif.Solver(**kw)
        s.upload(ux + h * dux, uy + h * duy, p)
        s.update_boundaries()
        q = {k: np.array(v, dtype=float) for k, v in parts.items()}
        for k, d in zip(("ux", "uy", "vz"), dvel):
            q[k] = q[k] + h * d
        s.set_particles(**q)
        return s

    h = 1e-6
    fd = (objective(solver(h), dts) - objective(solver(-h), dts)) / (2 * h)
    s = solver(0.0)
    s.tape_begin()
    for dt in dts:
        s.step_fixed_dt(dt, record=True)
    rec, w = s.particles(), 1.0 / len(dts)
    seed = np.zeros((1, 3))
    seed[:, 1] = -rec[:, 0] * np.pi * rec[:, 1] * rec[:, 2] * w
    for _ in dts:
        s.adjoint_add_wall_shear(w)
        s.adjoint_add(s.ADJ_FORCE, seed)
        for _ in range(3):
            s.stage_adjoint()
    terms = [s.adjoint_get(s.ADJ_UX) * dux, s.adjoint_get(s.ADJ_UY) * duy,
             s.adjoint_get(s.ADJ_PARTICLES)[0, 3:] * dvel]
    got = sum(float(t.sum()) for t in terms)
    scale = sum(float(np.abs(t).sum()) for t in terms)
    assert abs(got - fd) <= 1e-7 * scale, (got, fd, scale)
    halo = s.adjoint_get(s.ADJ_UX)
    assert not halo[0].any() and not halo[-1].any() and not halo[:, 0].any() and not halo[:, -1].any()
    halo = s.adjoint_get(s.ADJ_UY)
    assert not halo[0].any() and not halo[-1].any() and not halo[:, 0].any() and not halo[:, -1].any()


# box cells that make slices of 64, 128 and 256 cells (fewer than, about and
# more than 2048 waves), with a body across the periodic boundary; sums of up
# to 3e5 terms against the oracle's serial ones: 1e-12 of the largest member
@pytest.mark.parametrize("nx,n,a", [(64, 1, 0.1), (256, 300, 0.012), (512, 300, 0.016),
                                    (512, 300, 0.026)])
def test_slice_lengths(nx, n, a):
    ny = 2 * nx
    kw = dict(itot=nx, jtot=ny, ly=2.0, Re=100.0)
    g, o = eif.Solver(**kw), Oracle(**kw)
    ux, uy, p = cases.random_fields(nx, ny, 5)
    rng = np.random.default_rng(nx + n)
    y = rng.uniform(0, 2, n)
    y[0] = 1.999
    parts = dict(den=np.ones(n), a=np.full(n, a), b=np.full(n, 0.6 * a), x=rng.uniform(0.2, 0.8, n),
                 y=y, az=rng.uniform(0, 3, n))
    for s in (g, o):
        s.upload(ux, uy, p)
        s.update_boundaries()
        s.set_dt(1e-3)
        s.set_particles(**parts)
        s.reset_particle_increments()
        s.compute_inertia(0)
        s.exchange_momentum()
    x, y = g.particles()[:, 15:24], o.particles()[:, 15:24]
    assert np.max(np.abs(x - y)) <= 1e-12 * np.max(np.abs(y))
    g.close()


# partial sums of one and of several tiles of the diagnostics' second pass, and
# grids whose rows are shorter and longer than the stride: against numpy's
# pairwise sums, 1e-13 of the sum of magnitudes
@pytest.mark.parametrize("nx,ny", [(2, 3), (97, 33), (300, 700), (1024, 1024)])
def test_diagnostics_at_odd_sizes(nx, ny):
    s = eif.Solver(nx, ny, ly=1.5, Re=50.0)
    ux, uy, p = cases.random_fields(nx, ny, nx)
    s.upload(ux, uy, p)
    s.update_boundaries()
    f, g = s.download(), s.grid()
    u, v, dy = f["ux"][1:-1], f["uy"][1:-1, 1:-1], 1.5 / ny
    wx, wy = g["dxc"] * dy, g["dxf"] * dy
    div = (np.diff(u, axis=1) / g["dxf"]
           + (f["uy"][2:, 1:-1] - v) / dy)
    dmax, dsum = s.divergence()
    assert dmax == pytest.approx(np.max(np.abs(div)), rel=1e-13)
    assert abs(dsum - div.sum()) <= 1e-13 * np.abs(div).sum()
    for got, ref in ((s.momentum(), (u * wx, v * wy)),
                     (s.energy(), (0.5 * u * u * wx, 0.5 * v * v * wy))):
        for a, b in zip(got, ref):
            assert abs(a - b.sum()) <= 1e-13 * np.abs(b).sum()
    s.close()


# chunk counts of the partitioned solve: 2, ones that leave the matrix form's
# padding of 16 nearly empty or nearly full, its largest (192) and the lane
# loop past it, with a partial block of wavenumbers; psi less its mean against
# the sweep's within the conditioning of the line, about (jtot / pi)^2 eps
@pytest.mark.parametrize("nx,ny", [(20, 16), (16, 24), (32, 120), (33, 136), (64, 1024), (20, 1528),
                                   (16, 1544), (64, 8192)])
def test_partition_chunk_counts(nx, ny):
    ly = 4.0
    a, b = potential(nx, ny, ly, eif.POISSON_PARTITION)
    assert eif.partition_layout(ny)[1] >= 2
    a, b = a[1:-1, 1:-1], b[1:-1, 1:-1]
    a, b = a - a.mean(), b - b.mean()
    tol = max(1.0, (ny / np.pi) ** 2) * 2.3e-16 * 100
    assert np.linalg.norm(a - b) <= tol * np.linalg.norm(b)


# grids at which the predictor takes 2, 4, 8 and 16 rows a workgroup, with a
# partial last workgroup and a partial column block: whole stages (the kept
# previous velocity's form) and the per-function form, with the time step
@pytest.mark.parametrize("nx,ny", [(40, 27), (260, 1025), (260, 2050), (260, 4097)])
def test_predictor_rows_bit_exact(nx, ny):
    kw = dict(itot=nx, jtot=ny, ly=2.0, Re=100.0, extfrcy=0.1, uy_wall_xp=0.3)
    g, o = eif.Solver(**kw), Oracle(**kw)
    ux, uy, p = cases.random_fields(nx, ny, nx + ny, amp=0.3)
    for s in (g, o):
        s.upload(ux, uy, p)
        s.update_boundaries()
    assert g.decide_dt() == o.decide_dt()
    for s in (g, o):
        s.integrate()
    a, b = g.download(), o.download()
    for k in ("ux", "uy", "p"):
        assert np.array_equal(a[k], b[k]), k
    assert g.decide_dt() == o.decide_dt()
    for s in (g, o):
        s.update_velocity(0)
        s.update_velocity(1)
    a, b = g.download(), o.download()
    for k in ("ux", "uy"):
        assert np.array_equal(a[k], b[k]), k
    g.close()


# downloads through the staging slots: one slot (up to 2 MiB), a thread's
# strip of many chunks, several strips, with ragged ends; some fields left
# out; and into pinned memory, which is copied to directly
@pytest.mark.parametrize("nx,ny", [(6, 3), (300, 290), (301, 292), (500, 700), (1021, 1531)])
def test_downloads_return_the_fields(nx, ny):
    g = eif.Solver(nx, ny, ly=1.0)
    want = dict(zip(("ux", "uy", "p"), cases.random_fields(nx, ny, nx + ny)))
    g.upload(*want.values())
    for k, a in g.download().items():
        assert np.array_equal(a, want[k].reshape(a.shape)), k
    uy = np.full(g.shapes["uy"], -1.0)
    g._check(g.lib.fluid_gpu_download(g.h, None, eif._ptr(uy), None))
    assert np.array_equal(uy, want["uy"].reshape(uy.shape))
    p = torch.empty(g.shapes["p"], dtype=torch.float64, pin_memory=True).numpy()
    g._check(g.lib.fluid_gpu_download(g.h, None, None, eif._ptr(p)))
    assert np.array_equal(p, want["p"].reshape(p.shape))
    g.close()


# the cell list by one workgroup (up to 8192 particles, 1024 a turn) and by
# three launches: the partners of the test of all pairs, in the same order.
# Circles: the reference's fixed point of overlapping ellipses need not end.
@pytest.mark.parametrize("n", [1023, 1025, 8192, 8193])
def test_cell_list_finds_the_pairs_of_all_pairs(n):
    nx, ny, ly = 128, 256, 2.0
    k = np.arange(n)
    rng = np.random.default_rng(n)
    a = rng.uniform(0.007, 0.0085, n)
    part = dict(den=np.ones(n), a=a, b=a, x=(k % 64 + 0.5) / 64,
                y=(k // 64 + 0.5) * ly / 129, az=rng.uniform(0, 2 * np.pi, n), ux=np.zeros(n),
                uy=rng.uniform(-1, 1, n), vz=np.zeros(n))
    got = []
    for search in (eif.COLLISION_ALL_PAIRS, eif.COLLISION_CELLS):
        g = eif.Solver(nx, ny, ly=ly, poisson_mode=eif.POISSON_PARTITION)
        g.set_particles(**part)
        g.set_collision_search(search)
        g.compute_collision_force(0)
        got.append((g.colliding_pairs(), g.particles()))
        g.close()
    assert got[0][0] == got[1][0] and len(got[0][0]) > 20
    assert np.array_equal(got[0][1], got[1][1])


# weights of an ellipse 180 cells wide: distances past the exponential's
# clamp, its centre (foot on the evolute) and the saturated range.  The sums
# add 1.4e5 cells in another order than the oracle: at most N eps = 1.6e-11
# of the sum of the terms' sizes (positive here).
def test_inertia_of_a_wide_ellipse():
    kw = dict(itot=512, jtot=512, ly=1.0)
    part = dict(den=[1.0], a=[0.42], b=[0.36], x=[0.5], y=[0.5], az=[0.3])
    got = []
    for s in (eif.Solver(**kw), Oracle(**kw)):
        s.upload(ux=np.full(s.shapes["ux"], 0.75), uy=np.full(s.shapes["uy"], 1.25))
        s.update_boundaries()
        s.set_particles(**part)
        s.reset_particle_increments()
        s.compute_inertia(0)
        got.append(np.array(s.particles())[0])
        s.close()
    for m in (18, 20):  # iux, iuy of step 0
        assert got[1][m] > 0.5
        assert abs(got[0][m] - got[1][m]) <= 1.6e-11 * got[1][m]


# cell centres on the boundary of an ellipse whose axes are 325 and 65 cells
# (5 p, q cells from its centre, p^2 + q^2 = 65^2): there an error of the foot's
# parameter enters the distance linearly.  One velocity at a time reads the
# weights of two cells.  Ten roundings of coordinates below 0.5 are 6e-16, over
# the spacing of 1 / 1024 a distance of 6e-13 cells, and a weight changes by
# as much as the distance; from a cold start and from the foot of a body 1/64
# of a cell away.
@pytest.mark.parametrize("warm", [False, True])
def test_weights_on_the_boundary_of_a_thin_ellipse(warm):
    nx, ny, h = 1024, 512, 1.0 / 1024
    kw = dict(itot=nx, jtot=ny, ly=0.5, Re=100.0)
    a, b, shift = 325 * h, 65 * h, h / 64 if warm else 0.0
    part = dict(den=[1.0], a=[a], b=[b], x=[512.5 * h - shift], y=[256.5 * h], az=[0.0])
    legs = [(16, 63), (25, 60), (33, 56), (39, 52), (52, 39), (56, 33), (60, 25), (63, 16)]
    g, o = eif.Solver(**kw), Oracle(**kw)
    unit = 0.5 * h * h / (np.pi * a * b)
    zero = np.zeros(g.shapes["uy"])
    for s in (g, o):
        s.set_particles(**part)
        s.reset_particle_increments()
        if warm:
            s.compute_inertia(1)
            rec = s.particles()
            rec[:, 6] = shift
            s.set_particle_records(rec)
    for k, (p, q) in enumerate(legs):
        i, j = 513 + (5 * p if k & 1 else -5 * p), 257 + (q if k & 2 else -q)
        ux = np.zeros(g.shapes["ux"])
        ux[j, i - 1] = 1.0
        got = []
        for s in (g, o):
            s.upload(ux, zero)
            s.compute_inertia(1)
            got.append(s.particles()[0, 19] / unit)
        assert 0.4 < got[1] < 1.6
        assert abs(got[0] - got[1]) <= 2 * 6e-13, (p, q)
    g.close()


# a circle of 25 cells about a cell centre: twenty cell centres lie on its
# boundary, where the distance's gradient is the normal though the cell centre
# is its own foot.  The cotangent of the position against central differences,
# h = 1e-6: h^2 J''' is (128 h)^2 = 2e-8 of the derivative for weights that
# change over a cell of 1/128, round-off of the difference 1e-10 J
@pytest.mark.parametrize("az", [0.0, np.pi / 2])
def test_adjoint_of_a_body_with_cell_centres_on_its_boundary(az):
    n, h = 128, 1e-6
    kw = dict(itot=n, jtot=n, ly=1.0, Re=40.0, extfrcy=0.2)
    ux, uy, p = cases.random_fields(n, n, 3, amp=0.3)
    p[:] = 0.0
    c = 64.5 / n

    def solver(dx=0.0, dy=0.0):
        s = eif.Solver(**kw)
        s.upload(ux, uy, p)
        s.update_boundaries()
        s.set_particles(den=[1.3], a=[25.0 / n], b=[25.0 / n], x=[c + dx], y=[c + dy], az=[az],
                        ux=[0.1], uy=[-0.2], vz=[0.3])
        return s

    dts = [2e-4]
    fd = [(objective(solver(**{k: h}), dts) - objective(solver(**{k: -h}), dts)) / (2 * h)
          for k in ("dx", "dy")]
    s = solver()
    s.tape_begin()
    s.step_fixed_dt(dts[0], record=True)
    rec = s.particles()
    seed = np.zeros((1, 3))
    seed[:, 1] = -rec[:, 0] * np.pi * rec[:, 1] * rec[:, 2]
    s.adjoint_add_wall_shear(1.0)
    s.adjoint_add(s.ADJ_FORCE, seed)
    for _ in range(3):
        s.stage_adjoint()
    got = s.adjoint_get(s.ADJ_PARTICLES)[0, :2]
    assert np.max(np.abs(got - fd)) <= 1e-6 * np.max(np.abs(fd)), (got, fd)


# values that are no ordinary numbers, on a grid whose divisions are not by
# powers of two: an infinite, an overflowing and an undefined velocity give
# what the reference's divisions give (infinities stay infinite, and drive the
# time step to zero), and zeros keep their signs
@pytest.mark.parametrize("value", [np.inf, -np.inf, 1.7e308, np.nan, -0.0])
def test_grid_divisions_of_special_values(value):
    nx, ny = 48, 30
    kw = dict(itot=nx, jtot=ny, ly=0.9, Re=70.0)
    g, o = eif.Solver(**kw), Oracle(**kw)
    ux, uy, p = cases.random_fields(nx, ny, 9)
    psi = 0.1 * p
    if value == 0.0:
        for f in (ux, uy, p, psi):
            f[:] = 0.0
    for k, f in enumerate((ux, uy, p, psi)):
        f[11 + 3 * k, 17 + 2 * k] = value
    with np.errstate(all="ignore"):
        for s in (g, o):
            s.upload(ux, uy, p)
            s.update_boundaries()
        assert g.decide_dt() == o.decide_dt()
        for s in (g, o):
            s.set_dt(1e-3)
            s.update_velocity(0)
            s.set_field("psi", psi)
            s.correct_velocity(0)
            s.update_pressure()
        a, b = g.download(), o.download()
        for k in ("ux", "uy", "p"):
            assert np.array_equal(a[k], b[k], equal_nan=True), k
            there = ~np.isnan(a[k])
            assert np.array_equal(np.signbit(a[k][there]), np.signbit(b[k][there])), k
    g.close()


# bodies of 8.5 cells set to 10.9 cells by an upload of their records: their
# boxes of up to 900 cells fit the four slices of 256 made for 837, and have to
# fit shorter ones (14 of 64 cells would hold 896).  Sums of 4e5 terms against
# the oracle's serial ones, as for the slice lengths
@pytest.mark.parametrize("n", [1, 400])
def test_bodies_grown_by_their_records(n):
    nx, ny, h = 256, 512, 1.0 / 256
    kw = dict(itot=nx, jtot=ny, ly=2.0, Re=100.0)
    g, o = eif.Solver(**kw), Oracle(**kw)
    ux, uy, p = cases.random_fields(nx, ny, 5)
    rng = np.random.default_rng(n)
    parts = dict(den=np.ones(n), a=np.full(n, 8.5 * h), b=np.full(n, 8.5 * h),
                 x=rng.uniform(0.2, 0.8, n), y=rng.uniform(0.2, 1.8, n), az=rng.uniform(0, 3, n))
    parts["x"][0] = parts["y"][0] = 100.5 * h  # a box of 30 by 30
    for s in (g, o):
        s.upload(ux, uy, p)
        s.update_boundaries()
        s.set_dt(1e-3)
        s.set_particles(**parts)
        rec = s.particles()
        rec[:, 1:3] = 10.9 * h
        s.set_particle_records(rec)
        s.reset_particle_increments()
        s.compute_inertia(0)
        s.exchange_momentum()
        s.res = s.particles()[:, 15:24]
    g.synchronize()  # raises where a box did not fit
    assert np.max(np.abs(g.res - o.res)) <= 1e-12 * np.max(np.abs(o.res))
    g.close()


# downloads at the same time by six threads, more than there are sets of slots:
# from one context and from each thread's own, through one slot and in strips
@pytest.mark.parametrize("nx,ny", [(64, 96), (300, 290), (500, 700)])
@pytest.mark.parametrize("shared", [True, False])
def test_downloads_by_several_threads(nx, ny, shared):
    ss = [eif.Solver(nx, ny, ly=1.0) for _ in range(1 if shared else 6)]
    want = []
    for k, s in enumerate(ss):
        want.append(cases.random_fields(nx, ny, 31 * k + nx))
        s.upload(*want[-1])

    def work(t):
        s, w = ss[t % len(ss)], want[t % len(ss)]
        same = True
        for _ in range(6):
            d = s.download()
            same &= all(np.array_equal(d[k], f.reshape(d[k].shape)) for k, f in zip(("ux", "uy", "p"), w))
        return same

    with concurrent.futures.ThreadPoolExecutor(6) as pool:
        assert all(pool.map(work, range(6)))
    for s in ss:
        s.close()


# the slots are a device's, not a context's: downloads of 10 MB from 24 contexts
# one after the other, which need 4 MiB of slots, map less than 24 MiB (a set
# for each would be 96)
def test_downloads_of_many_contexts_share_their_slots():
    ss = [eif.Solver(512, 800, ly=1.0) for _ in range(24)]
    out = [np.zeros(ss[0].shapes[k]) for k in ("ux", "uy", "p")]

    def download(s):
        s._check(s.lib.fluid_gpu_download(s.h, *[eif._ptr(a) for a in out]))

    def mapped():
        with open("/proc/self/statm") as f:
            return int(f.read().split()[0]) * os.sysconf("SC_PAGE_SIZE")

    download(ss[0])
    before = mapped()
    for s in ss:
        download(s)
    assert mapped() - before < 24 << 20
    for s in ss:
        s.close()


def slice_length(nx, ny, ly, radii):
    """cells a slice, by the library's rule: 256, halved to 64 at least while
    the boxes make fewer than 2048 slices"""
    dx, dy = 1.0 / nx, ly / ny
    cells = 0
    for r in radii:
        wx, wy = min(int(2 * r / dx) + 10, nx), min(int(2 * r / dy) + 10, ny)
        cells += wx * (wy + 4) if ly > 2 * r + 16 * dy else 3 * wx * wy
    length = 256
    while length > 64 and cells // length < 2048:
        length //= 2
    return length


# slices of each length (100, 300 and 400 bodies of 1440 box cells), the
# distances searched from a cold start, served from the cache and searched from
# the last foot; sums of up to 6e5 terms against the oracle's serial ones:
# 1e-12 of the largest member
@pytest.mark.parametrize("n,length", [(100, 64), (300, 128), (400, 256)])
def test_slices_of_each_length(n, length):
    nx, ny, ly, a = 512, 1024, 2.0, 0.026
    assert slice_length(nx, ny, ly, [a] * n) == length
    kw = dict(itot=nx, jtot=ny, ly=ly, Re=100.0)
    g, o = eif.Solver(**kw), Oracle(**kw)
    ux, uy, p = cases.random_fields(nx, ny, 5)
    rng = np.random.default_rng(n)
    y = rng.uniform(0, 2, n)
    y[0] = 1.999
    parts = dict(den=np.ones(n), a=np.full(n, a), b=np.full(n, 0.6 * a), x=rng.uniform(0.2, 0.8, n),
                 y=y, az=rng.uniform(0, 3, n))
    for s in (g, o):
        s.upload(ux, uy, p)
        s.update_boundaries()
        s.set_dt(1e-3)
        s.set_particles(**parts)
        s.reset_particle_increments()
        s.compute_inertia(0)
        s.exchange_momentum()
        rec = s.particles()
        rec[:, 6:9] = [2e-4, -1e-4, 1e-3]
        s.set_particle_records(rec)
        s.compute_inertia(1)
    x, y = g.particles()[:, 15:24], o.particles()[:, 15:24]
    assert np.max(np.abs(x - y)) <= 1e-12 * np.max(np.abs(y))
    g.synchronize()
    g.close()
