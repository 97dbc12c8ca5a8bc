"""The learned initialiser's kernels at the sizes where their tiles end: the
staged convolution (strips of 64 x 1 and 32 x 2 voxels, rows and columns past
the volume, every channel split), the convolution of an upsampled and
concatenated input, the weight gradient (tiles, runs of planes, more units than
slices), and the elementwise kernels' scalar forms (channels and addresses that
16-byte accesses do not allow)."""
import ctypes as C
import os
import sys

import numpy as np
import pytest

from oracle import unet_ref as U
from timbir_amd.devmem import DevArray

sys.path.insert(0, os.path.dirname(os.path.abspath(__file__)))
from test_gpu_unet import bf, dev, empty, host, log, ptr  # noqa: E402

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def L():
    from timbir_amd import learned
    return learned.nn_lib()


def at(t, elems, size):
    """The address `elems` elements of `size` bytes into t."""
    return C.c_void_p(t.addr + elems * size)


@pytest.mark.parametrize("shape,cin,cout", [
    ((1, 1, 1, 1), 32, 32), ((1, 2, 9, 65), 32, 32), ((1, 3, 8, 64), 32, 96), ((2, 1, 5, 63), 64, 64),
    ((1, 2, 7, 33), 64, 32), ((1, 3, 4, 31), 96, 32), ((1, 2, 9, 40), 96, 64), ((1, 2, 5, 64), 128, 64),
    ((1, 2, 3, 20), 128, 128), ((1, 2, 10, 34), 192, 64), ((1, 1, 4, 66), 192, 192),
    ((1, 2, 3, 17), 160, 32)])   # 160: the kernel without LDS
def test_conv3d_tiles(L, shape, cin, cout):
    """fp32 output within 5e-5 of the largest value of the float64 result of
    the same bf16 operands (up to 27 x 192 fp32 products summed), as
    test_conv3d_matches_oracle; with bias and ReLU, and stored at an address
    that is not 16-byte aligned."""
    log(f"conv tile {shape} {cin}->{cout}")
    rng = np.random.default_rng(cin * 7 + cout)
    x = U.bf16(rng.standard_normal(shape + (cin,)).astype(np.float32))
    w = U.bf16((rng.standard_normal((27, cout, cin)) / np.sqrt(27 * cin)).astype(np.float32))
    b = rng.standard_normal(cout).astype(np.float32)
    xt, wt, bt, y = bf(x), bf(w), dev(b), empty((int(np.prod(shape)) * cout + 4,))
    ref = np.maximum(U.conv3d(x.astype(np.float64), w.astype(np.float64), b), 0)
    for off in (0, 1):
        assert L.tb_nn_conv3d(ptr(xt), ptr(wt), ptr(bt), at(y, off, 4), *shape, cin, cout, 1, 1,
                              None) == 0
        got = host(y)[off:off + ref.size].reshape(ref.shape)
        assert np.abs(got - ref).max() <= 5e-5 * np.abs(ref).max()


@pytest.mark.parametrize("shape,ca,cb,cout", [((1, 2, 2, 2), 64, 32, 32), ((2, 4, 10, 66), 64, 32, 32),
                                              ((1, 2, 8, 34), 64, 32, 64), ((1, 4, 6, 62), 128, 64, 64),
                                              ((1, 2, 18, 32), 128, 64, 96)])
def test_conv3d_up2cat_is_the_two_calls(L, shape, ca, cb, cout):
    """Bit for bit the upsampling and concatenation followed by the
    convolution; other channel counts are refused."""
    log(f"conv up2cat {shape} {ca}+{cb}->{cout}")
    rng = np.random.default_rng(ca + cout)
    n, d, h, w_ = shape
    a = bf(rng.standard_normal((n, d // 2, h // 2, w_ // 2, ca)))
    b = bf(rng.standard_normal(shape + (cb,)))
    w = bf(rng.standard_normal((27, cout, ca + cb)) / 30)
    bias = dev(rng.standard_normal(cout))
    cat, y1, y2 = (empty(shape + (c,), "bf16") for c in (ca + cb, cout, cout))
    assert L.tb_nn_up2_concat(ptr(a), ptr(b), ptr(cat), *shape, ca, cb, None) == 0
    assert L.tb_nn_conv3d(ptr(cat), ptr(w), ptr(bias), ptr(y1), *shape, ca + cb, cout, 1, 0, None) == 0
    assert L.tb_nn_conv3d_up2cat(ptr(a), ptr(b), ptr(w), ptr(bias), ptr(y2), *shape, ca, cb, cout, 1,
                                 None) == 0
    assert np.abs(host(y1)).max() > 0
    np.testing.assert_array_equal(host(y1), host(y2))
    assert L.tb_nn_conv3d_up2cat(ptr(a), ptr(b), ptr(w), ptr(bias), ptr(y2), *shape, 32, 32, cout, 1,
                                 None) == -1


@pytest.mark.parametrize("shape,cin,cout,slices", [
    ((1, 1, 1, 1), 32, 32, 1), ((1, 5, 16, 32), 32, 32, 3), ((2, 3, 17, 33), 32, 64, 256),
    ((1, 9, 15, 70), 96, 32, 5), ((3, 2, 33, 31), 64, 96, 2)])
@pytest.mark.parametrize("off", [0, 1])
def test_conv3d_wgrad_tiles(L, shape, cin, cout, slices, off):
    """Within 5e-5 of the largest value of the float64 sums, as
    test_conv3d_matches_oracle; operands at aligned and unaligned addresses."""
    log(f"wgrad tile {shape} {cin}->{cout} slices {slices} offset {off}")
    rng = np.random.default_rng(cin + 3 * cout)
    x = U.bf16(rng.standard_normal(shape + (cin,)).astype(np.float32))
    g = U.bf16(rng.standard_normal(shape + (cout,)).astype(np.float32))
    pad = np.zeros(off, np.float32)
    xt = bf(np.concatenate([pad, x.ravel()]))
    gt = bf(np.concatenate([pad, g.ravel()]))
    gw, part = empty((27, cout, cin)), empty((slices * 27 * cin * cout,))
    assert L.tb_nn_conv3d_wgrad(at(xt, off, 2), at(gt, off, 2), ptr(gw), ptr(part), slices, *shape,
                                cin, cout, None) == 0
    ref = U.conv3d_wgrad(x.astype(np.float64), g.astype(np.float64))
    assert np.abs(host(gw) - ref).max() <= 5e-5 * np.abs(ref).max()


@pytest.mark.parametrize("c,off", [(32, 0), (32, 1), (96, 0), (5, 0)])
def test_elementwise_forms_agree(L, c, off):
    """Pooling, upsampling, their backward passes, ReLU and the sum of two
    gradients in numpy on the same bf16 values, bit for bit; channel sums
    within 1e-5 of the sum of magnitudes (fp32 sums of a few hundred)."""
    log(f"elementwise c={c} offset {off}")
    rng = np.random.default_rng(c)
    shape = (2, 2, 4, 6)
    n, d, h, w = shape
    cell = (n, d // 2, h // 2, w // 2)
    x = U.bf16(rng.standard_normal(shape + (c,)).astype(np.float32))
    a = U.bf16(rng.standard_normal(cell + (c,)).astype(np.float32))

    def put(v):
        return bf(np.concatenate([np.zeros(off, np.float32), np.asarray(v, np.float32).ravel()]))

    def get(t, shp):
        return host(t)[off:].reshape(shp)

    def new(shp):
        return empty((int(np.prod(shp)) + off,), "bf16")

    def p(t):
        return at(t, off, 2)

    X, A = put(x), put(a)
    o = new(cell + (c,))
    assert L.tb_nn_avgpool2(p(X), p(o), *shape, c, 0, None) == 0
    s = np.zeros(cell + (c,), np.float32)
    for k in range(8):
        s = s + x[:, k >> 2::2, (k >> 1 & 1)::2, (k & 1)::2]
    np.testing.assert_array_equal(get(o, cell + (c,)), U.bf16(s * np.float32(0.125)))
    o = new(shape + (c,))
    assert L.tb_nn_avgpool2(p(A), p(o), *shape, c, 1, None) == 0
    np.testing.assert_array_equal(get(o, shape + (c,)), U.bf16(U.up2(a) * np.float32(0.125)))
    o = new(shape + (2 * c,))
    assert L.tb_nn_up2_concat(p(A), p(X), p(o), *shape, c, c, None) == 0
    np.testing.assert_array_equal(get(o, shape + (2 * c,)), np.concatenate([U.up2(a), x], -1))
    ga, gb = new(cell + (c,)), new(shape + (c,))
    cat = put(np.concatenate([x, U.up2(a)], -1))
    assert L.tb_nn_up2_concat_bwd(p(cat), p(ga), p(gb), *shape, c, c, None) == 0
    np.testing.assert_array_equal(get(ga, cell + (c,)), U.bf16(s))
    np.testing.assert_array_equal(get(gb, shape + (c,)), U.up2(a))
    y = put(-x)
    assert L.tb_nn_relu_bwd(p(X), p(y), x.size, None) == 0
    np.testing.assert_array_equal(get(y, x.shape), np.where(x > 0, -x, 0))
    z = put(U.up2(a))
    assert L.tb_nn_add(p(z), p(X), x.size, None) == 0
    np.testing.assert_array_equal(get(z, x.shape), U.bf16(U.up2(a) + x))
    for slices in (1, 7):
        out, part = empty((c,)), empty((slices * c,))
        nv = x.size // c
        assert L.tb_nn_channel_sum(p(X), ptr(out), ptr(part), slices, nv, c, None) == 0
        ref = x.reshape(nv, c).astype(np.float64)
        assert (np.abs(host(out) - ref.sum(0)) <= 1e-5 * np.abs(ref).sum(0)).all()


@pytest.mark.parametrize("c", [32, 64, 12])
def test_head_backward_and_network_input(L, c):
    """The head's gradients against numpy (the bf16 gradient bit for bit,
    the sums within 1e-5 of the sum of magnitudes), and the network input's
    channels for a mean shared by all samples."""
    log(f"head c={c}")
    rng = np.random.default_rng(c)
    nv, slices, scale = 333, 5, 50.0
    h = U.bf16(rng.standard_normal((nv, c)).astype(np.float32))
    w, g = (rng.standard_normal(k).astype(np.float32) for k in (c, nv))
    ht, wt, gt = bf(h), dev(w), dev(g)
    gh, part, hb = empty((nv, c), "bf16"), empty((slices, c + 1)), empty((c + 1,))
    assert L.tb_nn_head_bwd(ptr(ht), ptr(wt), ptr(gt), ptr(gh), ptr(part), slices, nv, c, scale,
                            None) == 0
    assert L.tb_nn_sum_parts(ptr(part), ptr(hb), c + 1, slices, None) == 0
    gs = (g * np.float32(1 / np.float32(scale))).astype(np.float32)
    np.testing.assert_array_equal(host(gh), U.bf16(gs[:, None] * w[None]))
    terms = np.concatenate([h, np.ones((nv, 1))], 1).astype(np.float64) * gs[:, None]
    assert (np.abs(host(hb) - terms.sum(0)) <= 1e-5 * np.abs(terms).sum(0)).all()
    per, v = 37, rng.standard_normal(3 * 37).astype(np.float32)
    m = rng.standard_normal(per).astype(np.float32)
    x = empty((v.size, 32), "bf16")
    assert L.tb_nn_make_input(ptr(dev(v)), ptr(dev(m)), ptr(x), v.size, per, scale, None) == 0
    want = np.zeros((v.size, 32), np.float32)
    want[:, 0] = U.bf16(v * np.float32(scale))
    want[:, 1] = U.bf16(np.tile(m, 3) * np.float32(scale))
    np.testing.assert_array_equal(host(x), want)


@pytest.mark.parametrize("shape", [(2, 3, 5, 7), (1, 1, 4, 6), (2, 4, 1, 3), (1, 2, 3, 1), (3, 5, 2, 2)])
@pytest.mark.parametrize("c,off", [(32, 0), (32, 1), (5, 0)])
def test_up2_concat_backward_of_odd_sizes(L, shape, c, off):
    """The skip connection's gradient at every voxel and the coarse one at the
    parents that odd sizes leave (their halves rounded down), bit for bit."""
    log(f"up2 concat backward {shape} c={c} offset {off}")
    rng = np.random.default_rng(c + shape[3])
    n, d, h, w = shape
    g = U.bf16(rng.standard_normal(shape + (2 * c,)).astype(np.float32))
    G = bf(np.concatenate([np.zeros(off, np.float32), g.ravel()]))
    cell = (n, d // 2, h // 2, w // 2, c)
    ga = bf(np.full(max(int(np.prod(cell)), 1) + off, 7.0))
    gb = bf(np.full(g.size // 2 + off, 7.0))
    assert L.tb_nn_up2_concat_bwd(at(G, off, 2), at(ga, off, 2), at(gb, off, 2), *shape, c, c,
                                  None) == 0
    np.testing.assert_array_equal(host(gb)[off:].reshape(shape + (c,)), g[..., c:])
    s = np.zeros(cell, np.float32)
    e = g[:, :d // 2 * 2, :h // 2 * 2, :w // 2 * 2, :c]
    for k in range(8):
        s = s + e[:, k >> 2::2, (k >> 1 & 1)::2, (k & 1)::2]
    np.testing.assert_array_equal(host(ga)[off:off + s.size].reshape(cell), U.bf16(s))


@pytest.mark.parametrize("shape,cin,cout", [((1, 3, 5, 20), 32, 32), ((2, 2, 9, 66), 32, 32),
                                            ((1, 2, 8, 33), 64, 64), ((1, 2, 4, 64), 96, 96),
                                            ((1, 2, 1, 40), 128, 64), ((1, 2, 17, 31), 192, 64)])
@pytest.mark.parametrize("value", [np.inf, np.nan])
def test_conv3d_leaves_out_taps_outside_the_volume(L, shape, cin, cout, value):
    """A weight that is infinite or NaN reaches only the voxels whose rows of
    that tap lie inside the volume: the staged convolution (and the one of a
    concatenation) gives the unstaged one's values, finite in the first and
    last rows where that is."""
    log(f"conv non-finite weight {shape} {cin}->{cout} {value}")
    rng = np.random.default_rng(cin + shape[2])
    n, d, h, w_ = shape
    x = bf(rng.standard_normal(shape + (cin,)))
    for dy in (0, 2):
        w = (rng.standard_normal((27, cout, cin)) / 30).astype(np.float32)
        w[dy * 3::9, 5, 7] = value
        wt, y = bf(w), empty((int(np.prod(shape)) * cout + 4,))
        got = []
        for off in (0, 1):
            assert L.tb_nn_conv3d(ptr(x), ptr(wt), None, at(y, off, 4), *shape, cin, cout, 0, 1,
                                  None) == 0
            got.append(host(y)[off:off + n * d * h * w_ * cout].reshape(shape + (cout,)))
        edge = got[1][:, :, 0 if dy == 0 else h - 1, :, 5]
        assert np.isfinite(edge).all()
        assert h == 1 or not np.isfinite(got[1][..., 5]).all()
        np.testing.assert_array_equal(got[0], got[1])


def test_conv3d_up2cat_leaves_out_taps_outside_the_volume(L):
    log("conv up2cat non-finite weight")
    rng = np.random.default_rng(3)
    for shape, ca, cb in (((1, 2, 6, 34), 64, 32), ((1, 4, 10, 66), 64, 32), ((1, 2, 6, 30), 128, 64)):
        n, d, h, w_ = shape
        a = bf(rng.standard_normal((n, d // 2, h // 2, w_ // 2, ca)))
        b = bf(rng.standard_normal(shape + (cb,)))
        w = (rng.standard_normal((27, 32, ca + cb)) / 30).astype(np.float32)
        w[0::9, 5, 7] = np.inf
        w[6::9, 9, ca + 3] = np.nan
        wt, bias, size = bf(w), dev(rng.standard_normal(32)), int(np.prod(shape)) * 32
        cat, y1, y2 = empty(shape + (ca + cb,), "bf16"), empty((size + 4,), "bf16"), empty((size,), "bf16")
        assert L.tb_nn_up2_concat(ptr(a), ptr(b), ptr(cat), *shape, ca, cb, None) == 0
        assert L.tb_nn_conv3d(ptr(cat), ptr(wt), ptr(bias), at(y1, 1, 2), *shape, ca + cb, 32, 1, 0,
                              None) == 0
        assert L.tb_nn_conv3d_up2cat(ptr(a), ptr(b), ptr(wt), ptr(bias), ptr(y2), *shape, ca, cb, 32,
                                     1, None) == 0
        want = host(y1)[1:size + 1].reshape(shape + (32,))
        assert np.isfinite(want[:, :, 0, :, 5]).all() and np.isfinite(want[:, :, -1, :, 9]).all()
        np.testing.assert_array_equal(host(y2).reshape(shape + (32,)), want)


def test_head_backward_without_slices_or_channels(L):
    """No slices: the activation gradient alone.  No channels: the bias
    gradient alone, its sums within 1e-5 of the sum of magnitudes."""
    log("head backward, slices 0 and c 0")
    rng = np.random.default_rng(5)
    for nv, c in ((700, 32), (333, 12)):
        h = U.bf16(rng.standard_normal((nv, c)).astype(np.float32))
        w, g = (rng.standard_normal(k).astype(np.float32) for k in (c, nv))
        ht, wt, gt = bf(h), dev(w), dev(g)
        gh, part = empty((nv, c), "bf16"), dev(np.full(4, 3.0))
        assert L.tb_nn_head_bwd(ptr(ht), ptr(wt), ptr(gt), ptr(gh), ptr(part), 0, nv, c, 4.0,
                                None) == 0
        np.testing.assert_array_equal(host(gh), U.bf16((g * np.float32(0.25))[:, None] * w[None]))
        np.testing.assert_array_equal(host(part), np.full(4, 3.0))
        part = empty((5, 1))
        assert L.tb_nn_head_bwd(None, None, ptr(gt), None, ptr(part), 5, nv, 0, 4.0, None) == 0
        assert abs(host(part).sum() - g.astype(np.float64).sum() / 4) <= 1e-5 * np.abs(g).sum() / 4


def test_network_of_other_widths_infers_as_it_trains(monkeypatch):
    """A network whose concatenations are not the 64 + 32 and 128 + 64 channels
    of tb_nn_conv3d_up2cat: its inference pass gives the training pass's
    output, bit for bit."""
    from timbir_amd import learned
    log("network of other widths")
    monkeypatch.setattr(learned, "ARCH", [
        ("e1a", "x", 32, 32), ("e1", "e1a", 32, 32), ("e2a", "pool:e1", 32, 32), ("e2", "e2a", 32, 32),
        ("b1", "pool:e2", 32, 96), ("b2", "b1", 96, 96), ("d2a", "cat:b2,e2", 128, 32),
        ("d2", "d2a", 32, 32), ("d1a", "cat:d2,e1", 64, 32), ("d1", "d1a", 32, 32)])
    monkeypatch.setattr(learned, "_LIVE", learned._live_sets())
    p = learned.init_params(3)
    rng = np.random.default_rng(3)
    p["head"] = (rng.normal(0, 0.1, 32).astype(np.float32), np.zeros(1, np.float32))
    net = learned.UNet(p)
    x = dev(rng.normal(0, 0.01, (2, 4, 8, 12)))
    a = net.forward(x, keep=True).numpy()
    b = net.forward(x).numpy()
    assert np.abs(a - x.numpy()).max() > 0
    np.testing.assert_array_equal(a, b)


@pytest.mark.parametrize("shape,c", [((1, 2, 2, 2), 8), ((3, 2, 2, 2), 40), ((1, 2, 2, 514), 8),
                                     ((64, 2, 6, 2), 16), ((1, 6, 10, 14), 24), ((1, 2, 258, 4), 3)])
def test_pooling_and_concatenation_of_narrow_volumes(L, shape, c):
    """Short rows, few rows, sides and channels of every kind of divisor:
    pooling, its backward pass and the concatenation, bit for bit."""
    log(f"pooling {shape} c={c}")
    rng = np.random.default_rng(c + shape[2])
    n, d, h, w = shape
    cell = (n, d // 2, h // 2, w // 2, c)
    x = U.bf16(rng.standard_normal(shape + (c,)).astype(np.float32))
    a = U.bf16(rng.standard_normal(cell).astype(np.float32))
    X, A, o, p, q = bf(x), bf(a), empty(cell, "bf16"), empty(x.shape, "bf16"), empty(shape + (2 * c,), "bf16")
    assert L.tb_nn_avgpool2(ptr(X), ptr(o), *shape, c, 0, None) == 0
    assert L.tb_nn_avgpool2(ptr(A), ptr(p), *shape, c, 1, None) == 0
    assert L.tb_nn_up2_concat(ptr(A), ptr(X), ptr(q), *shape, c, c, None) == 0
    s = np.zeros(cell, np.float32)
    for k in range(8):
        s = s + x[:, k >> 2::2, (k >> 1 & 1)::2, (k & 1)::2]
    np.testing.assert_array_equal(host(o), U.bf16(s * np.float32(0.125)))
    np.testing.assert_array_equal(host(p), U.bf16(U.up2(a) * np.float32(0.125)))
    np.testing.assert_array_equal(host(q), np.concatenate([U.up2(a), x], -1))


def test_pooling_of_more_rows_than_one_launch_has_blocks(L):
    """2^24 + 2 pooled rows of one voxel and channel."""
    log("pooling 2^24 rows")
    n = (1 << 24) + 2
    x = np.zeros((n, 8), np.float32)
    x[::7, 3] = 8.0
    x[-1] = 16.0
    X, o = bf(x), empty((n,), "bf16")
    assert L.tb_nn_avgpool2(ptr(X), ptr(o), n, 2, 2, 2, 1, 0, None) == 0
    np.testing.assert_array_equal(host(o), x.mean(1))


@pytest.mark.parametrize("cin", [32, 64, 96, 128, 192])
@pytest.mark.parametrize("cout", [32, 64, 96, 192])
@pytest.mark.parametrize("shape", [(1, 2, 5, 64), (197, 1, 8, 64), (195, 2, 9, 33), (130, 4, 1, 20),
                                   (23, 6, 3, 70)])
def test_conv3d_forms_give_the_same_bits(L, cin, cout, shape):
    """Launches small enough for 32 channels a wave, larger ones with 64 and 96
    and with two strips, and rows too few for the staged kernel: bit for bit
    the unstaged kernel's (the output stored at an odd address)."""
    log(f"conv forms {shape} {cin}->{cout}")
    rng = np.random.default_rng(cin + cout)
    x, w = bf(rng.standard_normal(shape + (cin,))), bf(rng.standard_normal((27, cout, cin)) / 30)
    bias, size = dev(rng.standard_normal(cout)), int(np.prod(shape)) * cout
    y1, y2 = empty((size,), "bf16"), empty((size + 8,), "bf16")
    assert L.tb_nn_conv3d(ptr(x), ptr(w), ptr(bias), ptr(y1), *shape, cin, cout, 0, 0, None) == 0
    assert L.tb_nn_conv3d(ptr(x), ptr(w), ptr(bias), at(y2, 1, 2), *shape, cin, cout, 0, 0, None) == 0
    assert np.abs(host(y1)).max() > 0
    np.testing.assert_array_equal(host(y1), host(y2)[1:size + 1])


@pytest.mark.parametrize("ca,cb", [(64, 32), (128, 64)])
@pytest.mark.parametrize("cout", [32, 64, 96])
@pytest.mark.parametrize("shape", [(2, 2, 6, 40), (100, 4, 6, 64), (70, 4, 10, 34), (150, 4, 2, 16)])
def test_conv3d_up2cat_forms_give_the_same_bits(L, ca, cb, cout, shape):
    log(f"conv up2cat forms {shape} {ca}+{cb}->{cout}")
    rng = np.random.default_rng(ca + cout)
    n, d, h, w_ = shape
    a = bf(rng.standard_normal((n, d // 2, h // 2, w_ // 2, ca)))
    b = bf(rng.standard_normal(shape + (cb,)))
    w, size = bf(rng.standard_normal((27, cout, ca + cb)) / 30), int(np.prod(shape)) * cout
    cat, y1, y2 = empty(shape + (ca + cb,), "bf16"), empty((size,), "bf16"), empty((size + 8,), "bf16")
    assert L.tb_nn_up2_concat(ptr(a), ptr(b), ptr(cat), *shape, ca, cb, None) == 0
    assert L.tb_nn_conv3d_up2cat(ptr(a), ptr(b), ptr(w), None, ptr(y1), *shape, ca, cb, cout, 1,
                                 None) == 0
    assert L.tb_nn_conv3d(ptr(cat), ptr(w), None, at(y2, 1, 2), *shape, ca + cb, cout, 1, 0, None) == 0
    np.testing.assert_array_equal(host(y1), host(y2)[1:size + 1])


@pytest.mark.parametrize("shape,cin,cout,slices", [
    ((3, 5, 1, 2), 32, 64, 4), ((40, 3, 2, 5), 64, 32, 7), ((1, 1, 1, 31), 96, 32, 256),
    ((2, 2, 3, 5), 32, 32, 1),                                       # 32 voxels at a time
    ((2, 5, 40, 70), 32, 32, 256), ((2, 4, 33, 66), 64, 96, 256), ((1, 9, 50, 31), 96, 32, 5),
    ((6, 3, 17, 65), 32, 64, 2)])                                    # in tiles
@pytest.mark.parametrize("off", [0, 1])
def test_conv3d_wgrad_of_narrow_and_of_large_volumes(L, shape, cin, cout, slices, off):
    """Either kernel of the weight gradient, to the bound of
    test_conv3d_wgrad_tiles."""
    test_conv3d_wgrad_tiles(L, shape, cin, cout, slices, off)


@pytest.mark.parametrize("n", [1, 63, 65, 32768, 32769, 131072, 131073, 200001])
@pytest.mark.parametrize("slices", [1, 7, 8, 16, 17, 70])
def test_sum_of_partial_sums(L, n, slices):
    """Every number of runs and their remainders: within 1e-6 of the sum of
    magnitudes of the float64 sums (at most 70 fp32 terms)."""
    log(f"sum parts n={n} slices={slices}")
    v = np.random.default_rng(n + slices).standard_normal((slices, n)).astype(np.float32)
    part, out = dev(v), empty((n,))
    assert L.tb_nn_sum_parts(ptr(part), ptr(out), n, slices, None) == 0
    want = v.astype(np.float64)
    assert (np.abs(host(out) - want.sum(0)) <= 1e-6 * np.abs(want).sum(0)).all()


@pytest.mark.parametrize("c", [8, 32, 200, 1024, 4200, 3, 70, 600])
@pytest.mark.parametrize("nv,slices", [(1, 1), (5, 9), (700, 2), (900, 300)])
def test_sums_over_voxels_of_any_width(L, c, nv, slices):
    """The bias gradient and the head's: channel groups of every size of a
    block and more than one block holds, more slices than voxels; within 1e-5
    of the sum of magnitudes, the activation gradient bit for bit."""
    log(f"channel sums c={c} nv={nv} slices={slices}")
    rng = np.random.default_rng(c + nv)
    x = U.bf16(rng.standard_normal((nv, c)).astype(np.float32))
    w, g = (rng.standard_normal(k).astype(np.float32) for k in (c, nv))
    xt, wt, gt, out, part = bf(x), dev(w), dev(g), empty((c,)), empty((slices * (c + 1),))
    assert L.tb_nn_channel_sum(ptr(xt), ptr(out), ptr(part), slices, nv, c, None) == 0
    ref = x.astype(np.float64)
    assert (np.abs(host(out) - ref.sum(0)) <= 1e-5 * np.abs(ref).sum(0)).all()
    gh, hb = empty((nv, c), "bf16"), empty((c + 1,))
    assert L.tb_nn_head_bwd(ptr(xt), ptr(wt), ptr(gt), ptr(gh), ptr(part), slices, nv, c, 2.0,
                            None) == 0
    assert L.tb_nn_sum_parts(ptr(part), ptr(hb), c + 1, slices, None) == 0
    gs = g * np.float32(0.5)
    np.testing.assert_array_equal(host(gh), U.bf16(gs[:, None] * w[None]))
    terms = np.concatenate([ref, np.ones((nv, 1))], 1) * gs[:, None].astype(np.float64)
    assert (np.abs(host(hb) - terms.sum(0)) <= 1e-5 * np.abs(terms).sum(0)).all()
