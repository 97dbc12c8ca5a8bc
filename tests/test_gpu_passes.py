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
