"""The multi-wavefront kernels' loads ahead of use: images so small that the
neighbours and records of a voxel are in flight while they are updated, voxel
lists shorter than a group, and entries at the generalized-Huber threshold,
where the rounded decision hands over to the exact one."""
import os
import sys

import numpy as np
import pytest

import timbir_amd as tb
from oracle import pyorc
from timbir_amd import datagen

sys.path.insert(0, os.path.dirname(os.path.abspath(__file__)))
from test_gpu_parity import check_kernel  # noqa: E402

pytestmark = pytest.mark.gpu


@pytest.fixture(params=[3, 4, 8, 0], ids=["multiwave", "mwglobal", "mwdeep", "auto"])
def kernel(request):
    old = tb.get_options()
    tb.set_options(kernel=request.param)
    yield request.param
    tb.set_options(kernel=old.kernel, hicd_order=old.hicd_order)


@pytest.mark.parametrize("raster", [0, 1])
@pytest.mark.parametrize("N,nz,n_views", [(4, 2, 8), (5, 3, 11), (8, 4, 43), (11, 3, 86)])
def test_voxels_in_flight(kernel, raster, N, nz, n_views):
    """Whole sweeps of images of 4 to 11 pixels a side (chunks of 1 to 12
    voxels, nearly every neighbour in flight) in shuffled and raster order
    against the oracle's same schedule: a stale neighbour or entry is wrong
    by a step (of the order of the object), rounding by 1e-6 of the range;
    the bound is the trajectory tests' 1e-4."""
    print(f"in flight N={N} nz={nz} views={n_views} raster={raster} kernel={kernel}", flush=True)
    scan = datagen.tiny(N=N, nz=nz, n_frames=2, n_views=n_views, sig_s=0.005, sig_t=0.01,
                        convg_thresh=0.0, quad_convex=0, zingers=1e-2, c_s=1.0, c_t=1.0)
    tb.set_options(hicd_order=raster)
    o = pyorc.Problem(scan, opt=pyorc.options(schedule=pyorc.SCHED_COLOUR, hicd_order=raster))
    g = tb.Stage(scan)
    o.init_error_sino()
    g.init_error_sino()
    for it in range(1, 4):
        o.icd_iteration(it)
        g.icd_iteration(it)
        xo, xg = o.obj(), g.object()
        rmse = np.sqrt(np.mean((xg - xo) ** 2)) / (xo.max() - xo.min())
        assert rmse < 1e-4, (it, rmse)
        eo, eg = o.err(), g.error_sino()
        assert np.abs(eg - eo).max() <= 1e-4 * np.abs(eo).max()
    g.close()


@pytest.mark.parametrize("kern", [3, 4])
@pytest.mark.parametrize("T", [1.5, np.nextafter(np.float32(1.5), np.float32(2)),
                               np.nextafter(np.float32(1.5), np.float32(1)),
                               1.5 * (1 + 2.0 ** -19), 1.5 * (1 - 2.0 ** -19), 1.49, 1.51])
def test_huber_threshold(kern, T):
    """Every entry has |e sqrt(w)| = 1.5 exactly: at T = 1.5 and the float
    below none is inside, at the float above all are, and so on through the
    band's edges.  A wrong side changes the step by the threshold's factor
    delta = 0.5; the single update's tolerance is 2e-5 of it."""
    print(f"huber threshold T={float(T)!r} kernel={kern}", flush=True)
    scan = datagen.tiny(N=16, nz=2, n_frames=1, n_views=24, sig_s=0.005, sig_t=0.01,
                        quad_convex=0, c_s=1.0, c_t=1.0)
    scan["projections"] = np.full_like(scan["projections"], 0.75)
    scan["weights"] = np.full_like(scan["weights"], 4.0)
    scan["huber_T"] = float(np.float32(T))
    old = tb.get_options().kernel
    tb.set_options(kernel=kern)
    try:
        o = pyorc.Problem(scan, opt=pyorc.options(schedule=pyorc.SCHED_COLOUR))
        g = tb.Stage(scan)
        o.init_error_sino()
        g.init_error_sino()
        vo = o.voxel_update(0, 1, 8, 8)
        vg = g.voxel_update(0, 1, 8, 8)
        assert abs(vg - vo) <= 2e-5 * abs(vo), (vg, vo)
        g.close()
    finally:
        tb.set_options(kernel=old)


@pytest.mark.parametrize("raster", [0, 1])
@pytest.mark.parametrize("kern,N,nz,views,mult", [
    (4, 4, 2, 400, (1, 1)), (4, 8, 2, 700, (1, 1)),                            # records RD 2: 2 and 4 views a lane
    (4, 10, 4, 90, (2, 2)), (4, 16, 4, 170, (2, 2)), (4, 8, 4, 300, (2, 2)),   # 5 bins x 2 rows, 15 slots, 2 views
    (4, 16, 8, 100, (4, 4)), (4, 20, 8, 180, (4, 4)), (4, 24, 4, 90, (4, 2)),  # 9 bins x 4 rows: RD 4; 2 rows
    (3, 10, 4, 40, (2, 2)), (3, 22, 4, 90, (2, 2)), (0, 16, 8, 60, (4, 4))])
def test_voxels_in_flight_of_wide_columns(kern, N, nz, views, mult, raster):
    """test_voxels_in_flight for the record rings of two and four records, the
    columns of several rows, several views a lane and the exchange of 15 slots:
    lists shorter than the rings, to the same bounds."""
    print(f"in flight N={N} nz={nz} views={views} mult={mult} raster={raster} kernel={kern}", flush=True)
    scan = datagen.tiny(N=N, nz=nz, n_frames=2, n_views=2 * views, sig_s=0.005, sig_t=0.01,
                        convg_thresh=0.0, quad_convex=0, c_s=1.0, c_t=1.0)
    old = tb.get_options()
    tb.set_options(hicd_order=raster, kernel=kern)
    try:
        o = pyorc.Problem(scan, mult_xy=mult[0], mult_z=mult[1],
                          opt=pyorc.options(schedule=pyorc.SCHED_COLOUR, hicd_order=raster))
        g = tb.Stage(scan, mult_xy=mult[0], mult_z=mult[1])
        o.init_error_sino()
        g.init_error_sino()
        for it in range(1, 4):
            o.icd_iteration(it)
            g.icd_iteration(it)
            xo, xg = o.obj(), g.object()
            rmse = np.sqrt(np.mean((xg - xo) ** 2)) / (xo.max() - xo.min())
            assert rmse < 1e-4, (it, rmse)
            eo, eg = o.err(), g.error_sino()
            assert np.abs(eg - eo).max() <= 1e-4 * np.abs(eo).max()
        check_kernel(g, kern)
        g.close()
    finally:
        tb.set_options(kernel=old.kernel, hicd_order=old.hicd_order)


@pytest.mark.parametrize("kern", [2, 3, 4, 8])
@pytest.mark.parametrize("seed", [0, 1, 2])
@pytest.mark.parametrize("side", [-1, 1])
def test_huber_side_inside_the_band(kern, seed, side):
    """Products that round, e^2 w off T^2 by 2.5e-7 to 9e-7 of it: inside the
    rounded decision's band and four times outside what huber_sel may err by
    (2^-24).  Every entry takes its side, to the tolerance above."""
    from fractions import Fraction
    rng = np.random.default_rng(seed)
    while True:
        T, e = np.float32(rng.uniform(1, 5)), np.float32(rng.uniform(0.05, 0.5))
        w = np.float32(float(T) ** 2 / float(e) ** 2 * (1 + side * rng.uniform(2.5e-7, 9e-7)))
        off = Fraction(float(e)) ** 2 * Fraction(float(w)) / Fraction(float(T)) ** 2 - 1
        if 2.5e-7 <= side * off <= 9e-7 and Fraction(float(e)) ** 2 != Fraction(float(e * e)):
            break
    print(f"huber band e={e!r} w={w!r} T={T!r} off={float(off):.2e} kernel={kern}", flush=True)
    scan = datagen.tiny(N=16, nz=2, n_frames=1, n_views=24, sig_s=0.005, sig_t=0.01,
                        quad_convex=0, c_s=1.0, c_t=1.0)
    scan["projections"] = np.full_like(scan["projections"], e)
    scan["weights"] = np.full_like(scan["weights"], w)
    scan["huber_T"] = float(T)
    old = tb.get_options().kernel
    tb.set_options(kernel=kern)
    try:
        o = pyorc.Problem(scan, opt=pyorc.options(schedule=pyorc.SCHED_COLOUR))
        g = tb.Stage(scan)
        o.init_error_sino()
        g.init_error_sino()
        vo = o.voxel_update(0, 1, 8, 8)
        vg = g.voxel_update(0, 1, 8, 8)
        assert abs(vg - vo) <= 2e-5 * abs(vo), (vg, vo)
        check_kernel(g, kern)
        g.close()
    finally:
        tb.set_options(kernel=old)
