"""The passes around the voxel kernels at the sizes where they can go wrong:
the filtered back-projection (slice groups, odd detector widths, a rotation
axis off centre, so that rays miss the detector), the prior cost (differences
at the ends of FP32's range, edges of the volume) and the forward projector
(a lone slice, a partial group, an off-centre axis)."""
import os
import sys

import numpy as np
import pytest

import timbir_amd as tb
from timbir_amd import datagen

sys.path.insert(0, os.path.dirname(os.path.abspath(__file__)))
import mathref  # noqa: E402
from test_fbp import stage_fbp_reference  # noqa: E402

pytestmark = pytest.mark.gpu


def scan_of(N, nz, rot_shift=0.0, n_frames=2, n_views=22, **kw):
    s = datagen.tiny(N=N, nz=nz, n_frames=n_frames, n_views=n_views, **kw)
    s["rot_center"] = N / 2 + rot_shift
    return s


@pytest.mark.parametrize("N,nz,shift", [(16, 1, 0.0), (17, 3, 0.0), (33, 4, 2.5), (31, 5, -3.0),
                                        (40, 8, 0.5), (26, 9, 7.0), (64, 17, 0.0)])
def test_fbp_groups_and_edges(N, nz, shift):
    """Within 1e-5 of the largest value of the FP64 numpy statement (the
    output is FP32, its sums FP64), for every remainder of the slice groups
    and of the filter's output groups."""
    print(f"fbp N={N} nz={nz} shift={shift}", flush=True)
    scan = scan_of(N, nz, shift)
    st = tb.Stage(scan)
    off = np.random.default_rng(4).normal(0, 0.01, (N, nz)).astype(np.float32)
    st.set_offset(off)
    st.init_fbp()
    got = st.object()
    ref = stage_fbp_reference(scan, st, off)
    st.close()
    assert np.abs(ref).max() > 0
    np.testing.assert_allclose(got, ref, rtol=0, atol=1e-5 * np.abs(ref).max())


@pytest.mark.parametrize("scale", [0.0, 1e-42, 1e-30, 1e-12, 1.0, 1e12, 1e20])
@pytest.mark.parametrize("shape", [(1, 1, 5), (2, 3, 17), (3, 2, 19)])
def test_prior_cost_over_the_float_range(scale, shape):
    """The prior cost against its numpy statement in FP64 (mathref.rho over
    the forward neighbour pairs) within 1e-12: both sum FP64 terms of a few
    rounding errors each."""
    print(f"prior cost scale={scale} shape={shape}", flush=True)
    F, Z, N = shape
    scan = scan_of(N, Z, n_frames=F, n_views=6 * F, c_s=1e-2, c_t=1e-2)
    st = tb.Stage(scan)
    rng = np.random.default_rng(8)
    x = rng.normal(0, 1, st.obj_shape).astype(np.float32)
    x[..., ::3] = 0.0                       # zero differences among them
    x = (x * np.float32(scale)).astype(np.float32)
    st.set_object(x)
    got = st.cost()[2]
    i, f = st.info, st.sfilt
    st.close()
    xd = x.astype(np.float64)
    ref = 0.0
    for dz in (0, 1):
        for dy in (-1, 0, 1):
            for dx in (-1, 0, 1):
                if (dz, dy, dx) <= (0, 0, 0):
                    continue
                a = xd[:, :Z - dz, max(0, -dy):N - max(0, dy), max(0, -dx):N - max(0, dx)]
                b = xd[:, dz:, max(0, dy):N - max(0, -dy), max(0, dx):N - max(0, -dx)]
                ref += f[dz + 1, dy + 1, dx + 1] * mathref.rho(a - b, i["sigS_q"], i["sigS_qp"],
                                                               i["c_s"]).sum()
    ref += i["tfilt"] * mathref.rho(xd[:-1] - xd[1:], i["sigT_q"], i["sigT_qp"], i["c_t"]).sum()
    assert abs(got - ref) <= 1e-12 * abs(ref), (got, ref)


def test_prior_cost_keeps_infinities_and_nan():
    scan = scan_of(16, 2, n_frames=1, n_views=8)
    st = tb.Stage(scan)
    x = np.zeros(st.obj_shape, np.float32)
    st.set_object(x)
    assert st.cost()[2] == 0.0
    x[0, 1, 5, 5] = np.nan
    st.set_object(x)
    assert np.isnan(st.cost()[2])
    st.close()


@pytest.mark.parametrize("N,nz,shift,mxy,mz", [(15, 1, 0.0, 1, 1), (18, 5, 1.25, 1, 1),
                                               (20, 4, -4.0, 2, 2), (24, 12, 0.0, 1, 1),
                                               (24, 8, 3.0, 4, 4)])
def test_forward_projection_bitwise_at_the_edges(N, nz, shift, mxy, mz):
    """Bit for bit the oracle's forward projection, as
    test_forward_projection_bitwise asserts on a centred scan."""
    from oracle import pyorc
    print(f"forward N={N} nz={nz} shift={shift} mult={mxy},{mz}", flush=True)
    scan = scan_of(N, nz, shift, n_views=34)
    st = tb.Stage(scan, mult_xy=mxy, mult_z=mz)
    o = pyorc.Problem(scan, mult_xy=mxy, mult_z=mz)
    x = np.random.default_rng(6).random(st.obj_shape).astype(np.float32)
    st.set_object(x)
    o.obj()[...] = x
    got = st.forward_project()
    st.close()
    np.testing.assert_array_equal(got, o.forward_project())
    assert np.abs(got).max() > 0


@pytest.mark.parametrize("kind", ["ties", "wide"])
@pytest.mark.parametrize("N", [3, 8, 16, 90, 91, 128, 129, 181, 182, 200])
def test_line_selection_at_its_register_limits(N, kind):
    """NHICD line lists of cells of 9 to 40000 pixels (a cell's pixels in 8,
    16 or 32 registers a lane up to 90, 128 and 181 pixels a side, read again
    beyond; ragged last steps) hold the order statistic of the filtered map: the
    (N^2 - want)-th smallest is the threshold and the lines above it follow in
    raster order, as the oracle's lists, entry for entry."""
    from oracle import pyorc
    print(f"line selection N={N} {kind}", flush=True)
    s = datagen.tiny(N=N, nz=2, n_frames=1, n_views=4)
    o = pyorc.Problem(s, opt=pyorc.options(schedule=pyorc.SCHED_COLOUR))
    g = tb.Stage(s)
    rng = np.random.default_rng(N)
    mag = rng.random(o.obj_shape).astype(np.float32)
    if kind == "ties":
        mag = np.floor(mag * 2).astype(np.float32)
        mag[..., : N // 2, :] = 0.0
    else:
        mag = np.exp(-60.0 * mag).astype(np.float32)
    o.mag()[...] = mag
    g.set_magmap(mag)
    o.L.orc_set_select_counts(o.h, o.info["U"])
    o.vsc_select()
    g.vsc_select()
    for z in range(o.info["N_z"]):
        xo, yo = o.nhicd_list(0, z)
        xg, yg = g.nhicd_list(0, z)
        np.testing.assert_array_equal(xg, xo)
        np.testing.assert_array_equal(yg, yo)
    # the selection clears the map at selected pixels outside the mask (the
    # oracle does when it reaches them) and nowhere else
    changed = g.magmap() != mag
    assert not changed[..., o.mask() == 1].any() and not g.magmap()[changed].any()
    g.close()


@pytest.mark.parametrize("N,nz,shift", [(23, 2, 0.0), (30, 6, -1.5), (21, 7, 4.0), (18, 10, 0.0),
                                        (25, 15, 2.0), (32, 16, 0.0)])
def test_fbp_of_a_groups_remainder(N, nz, shift):
    """The numbers of slices in the last group that test_fbp_groups_and_edges
    has not, each its own kernel and row stride, to the same bound."""
    test_fbp_groups_and_edges(N, nz, shift)


@pytest.mark.parametrize("where", ["one", "pair", "ends"])
def test_prior_cost_at_infinities_and_the_largest_values(where):
    """The numpy statement's value where the fast form's FP32 range ends: a
    difference with an infinity and of two infinities (both NaN there), and of
    the largest finite values of either sign (within 1e-12, as above)."""
    print(f"prior cost {where}", flush=True)
    scan = scan_of(9, 2, n_frames=2, n_views=12)
    st = tb.Stage(scan)
    x = np.random.default_rng(2).normal(0, 1, st.obj_shape).astype(np.float32)
    if where == "ends":
        x = (np.sign(x) * np.finfo(np.float32).max).astype(np.float32)
    else:
        x[0, 1, 4, 4] = np.inf
        if where == "pair":
            x[0, 1, 4, 5] = np.inf
    st.set_object(x)
    got = st.cost()[2]
    i, f = st.info, st.sfilt
    st.close()
    with np.errstate(invalid="ignore", over="ignore"):
        xd, ref = x.astype(np.float64), 0.0
        for dz, dy, dx in [(a, b, c) for a in (0, 1) for b in (-1, 0, 1) for c in (-1, 0, 1)
                           if (a, b, c) > (0, 0, 0)]:
            a = xd[:, :2 - dz, max(0, -dy):9 - max(0, dy), max(0, -dx):9 - max(0, dx)]
            b = xd[:, dz:, max(0, dy):9 - max(0, -dy), max(0, dx):9 - max(0, -dx)]
            ref += f[dz + 1, dy + 1, dx + 1] * mathref.rho(a - b, i["sigS_q"], i["sigS_qp"],
                                                           i["c_s"]).sum()
        ref += i["tfilt"] * mathref.rho(xd[:-1] - xd[1:], i["sigT_q"], i["sigT_qp"], i["c_t"]).sum()
    if where == "ends":
        assert np.isfinite(ref) and abs(got - ref) <= 1e-12 * abs(ref), (got, ref)
    else:
        assert np.isnan(ref) and np.isnan(got), (got, ref)


def test_fbp_of_more_frames_than_one_launch_has_blocks():
    """2^24 + 3 frames of 4 x 4 pixels, the views all in frame 2^24 - 1: its
    back-projection stands there, equal to that of one such frame alone, and
    every other frame is zero."""
    print("fbp of 2^24 frames", flush=True)
    F, at = (1 << 24) + 3, (1 << 24) - 1
    one = datagen.tiny(N=4, nz=1, n_frames=1, n_views=8)
    st = tb.Stage(one)
    st.init_fbp()
    want = st.object()
    st.close()
    many = dict(one, recon_num=F, recon_times=np.arange(F + 1, dtype=np.float64).astype(np.float32),
                proj_times=np.full(8, at, np.float32))
    st = tb.Stage(many)
    st.init_fbp()
    got = st.object()
    st.close()
    assert np.abs(want).max() > 0
    np.testing.assert_array_equal(got[at], want[0])
    got[at] = 0.0
    assert not got.any()
