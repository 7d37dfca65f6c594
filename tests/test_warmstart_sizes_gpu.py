"""The warm-start network's layers away from the square images of the network:
sizes of nothing, images of few rows or columns, arrays past 32-bit offsets."""
import ctypes

import numpy as np
import pytest

from mplb_amd import warmstart as ws
from oracle import nn_oracle as nno

pytestmark = pytest.mark.gpu


def log(m):
    print(m, flush=True)


def ck(rc):
    assert rc == 0, rc


def at(d, offset):
    """Element `offset` of a device array."""
    return ctypes.c_void_p(d.p.value + 4 * offset)


# no image, no row, no column, no channel; all that is none is negative too
@pytest.mark.parametrize("n,h,wd,c", [(0, 2, 2, 4), (2, 0, 2, 4), (2, 2, 0, 4), (2, 2, 2, 0),
                                      (-1, 2, 2, 4), (2, -2, 2, 4), (2, 2, -2, 4), (2, 2, 2, -4),
                                      (2, 2, 2, -3)])
def test_upsampling_and_channel_copies_of_nothing(n, h, wd, c):
    log("nothing %s" % ((n, h, wd, c),))
    lib, rng = ws.load(), np.random.default_rng(3)
    a, b = (rng.standard_normal((2, 4, 4, 8)).astype(np.float32) for _ in range(2))
    da, db = ws.DeviceArray.from_numpy(a), ws.DeviceArray.from_numpy(b)
    ck(lib.mplbws_up2_fwd(da.p, db.p, n, h, wd, c, 8, 0))
    ck(lib.mplbws_up2_bwd(da.p, db.p, n, h, wd, c, 8, 0))
    for direction in range(3):
        ck(lib.mplbws_channels(da.p, db.p, n * h * wd, c, 8, 0, direction)
           if c <= 0 or n * h * wd <= 0 else 0)
    assert np.array_equal(da.numpy(), a) and np.array_equal(db.numpy(), b)


# one row, one column, more channels than pixels; an index past 2^30 items
@pytest.mark.parametrize("rows,wd,c,ctot,c0", [(1, 3000, 16, 24, 8), (3000, 1, 5, 7, 1),
                                               (1, 1, 20000, 20004, 4), (2, 3, 1031, 1031, 0)])
def test_upsampling_and_channel_copies_of_thin_images(rows, wd, c, ctot, c0):
    log("thin %s" % ((rows, wd, c, ctot, c0),))
    lib, rng = ws.load(), np.random.default_rng(4)
    A = ws.DeviceArray.from_numpy
    x = rng.standard_normal((1, rows, wd, c)).astype(np.float32)
    wide = rng.standard_normal((1, 2 * rows, 2 * wd, ctot)).astype(np.float32)
    dx, dw = A(x), A(wide)
    ck(lib.mplbws_up2_fwd(dx.p, dw.p, 1, rows, wd, c, ctot, c0))
    ref = wide.copy()
    ref[..., c0:c0 + c] = x.repeat(2, axis=1).repeat(2, axis=2)
    assert np.array_equal(dw.numpy(), ref)
    dw = A(wide)
    ck(lib.mplbws_up2_bwd(dw.p, dx.p, 1, rows, wd, c, ctot, c0))
    f = wide[..., c0:c0 + c]
    assert np.array_equal(dx.numpy(), (f[:, ::2, ::2] + f[:, ::2, 1::2])
                          + (f[:, 1::2, ::2] + f[:, 1::2, 1::2]))
    thin = ws.DeviceArray((1, 2 * rows, 2 * wd, c))
    ck(lib.mplbws_channels(dw.p, thin.p, 4 * rows * wd, c, ctot, c0, 1))
    assert np.array_equal(thin.numpy(), f)


def test_upsampling_and_channel_copies_past_two_to_the_thirty_items():
    """One channel, so an item per pixel: the last pixels of 2^30 + 4096, in a
    few long rows and in many short ones."""
    lib, rng = ws.load(), np.random.default_rng(6)
    total, tail = (1 << 30) + 4096, 256
    v = rng.standard_normal(tail).astype(np.float32)
    coarse, fine = ws.DeviceArray((total,)), ws.DeviceArray((4 * total,))

    def put(d, offset, a):
        ck(lib.mplbws_upload(at(d, offset), a.ctypes.data, a.nbytes))

    def get(d, offset, count):
        out = np.empty(count, np.float32)
        ck(lib.mplbws_download(out.ctypes.data, at(d, offset), out.nbytes))
        return out

    for rows in (1, total // 4096):
        log("up %d x %d" % (rows, total // rows))
        wd = total // rows
        put(coarse, total - tail, v)
        ck(lib.mplbws_zero(fine.p, 4 * fine.numel()))
        ck(lib.mplbws_up2_fwd(coarse.p, fine.p, 1, rows, wd, 1, 1, 0))
        for row in (1, 2):  # the last two fine rows
            end = 4 * total - (row - 1) * 2 * wd
            assert np.array_equal(get(fine, end - 2 * tail, 2 * tail), v.repeat(2))
        put(coarse, total - tail, np.zeros(tail, np.float32))
        ck(lib.mplbws_up2_bwd(fine.p, coarse.p, 1, rows, wd, 1, 1, 0))
        assert np.array_equal(get(coarse, total - tail, tail), 4 * v)
    put(coarse, total - tail, np.zeros(tail, np.float32))
    put(fine, total - tail, v)
    ck(lib.mplbws_channels(fine.p, coarse.p, total, 1, 1, 0, 1))
    assert np.array_equal(get(coarse, total - tail, tail), v)


# one to seven rows, in tiles of more than 32 columns: one column short of a
# tile, a tile, several with a remainder, and enough images for larger tiles
@pytest.mark.parametrize("n,h,wd,cin,cout", [(1, 1, 66, 8, 4), (2, 1, 67, 16, 8), (530, 1, 111, 8, 4),
                                             (2, 2, 99, 8, 33), (1, 3, 39, 40, 8),
                                             (300, 2, 166, 8, 8), (1, 5, 101, 8, 5),
                                             (3, 7, 70, 24, 24)])
def test_convolution_of_few_rows(n, h, wd, cin, cout):
    log("conv %s" % ((n, h, wd, cin, cout),))
    lib, rng = ws.load(), np.random.default_rng(11)
    A = ws.DeviceArray.from_numpy
    x = rng.standard_normal((n, h, wd, cin)).astype(np.float32)
    w = (rng.standard_normal((9, cin, cout)) / 8).astype(np.float32)
    dx, dw, out = A(x), A(w), ws.DeviceArray((n, h, wd, cout))
    ck(lib.mplbws_conv3x3_fwd(dx.p, dw.p, None, out.p, n, h, wd, cin, cout, 0))
    # FP32 sums of 9 cin exact products
    tol = (9 * cin + 1) * 2.0 ** -24 * nno.conv3x3(np.abs(x), np.abs(w))
    assert (np.abs(out.numpy() - nno.conv3x3(x, w)) <= tol).all()


# few columns (taken along them), two chunks of one and of nine, few rows in
# long lines, and channel counts that are no multiple of four on either side
@pytest.mark.parametrize("n,h,wd,cin,cout", [(1, 300, 1, 8, 4), (2, 130, 2, 5, 3), (1, 97, 3, 33, 12),
                                             (3, 40, 7, 8, 67), (1, 5000, 1, 4, 4),
                                             (1, 700, 9, 12, 8), (1, 1, 200, 8, 8),
                                             (1, 2, 150, 6, 5), (2, 33, 33, 40, 35),
                                             (2, 33, 33, 39, 36), (1, 20, 20, 1, 1)])
def test_weight_gradient_of_thin_images_and_odd_channels(n, h, wd, cin, cout):
    log("wgrad %s" % ((n, h, wd, cin, cout),))
    lib, rng = ws.load(), np.random.default_rng(13)
    A = ws.DeviceArray.from_numpy
    x = rng.standard_normal((n, h, wd, cin)).astype(np.float32)
    d = rng.standard_normal((n, h, wd, cout)).astype(np.float32)
    dw, db = ws.DeviceArray((9, cin, cout)), ws.DeviceArray((cout,))
    k = ws.DeviceArray((int(lib.mplbws_wgrad_workspace(n, h, wd, cin, cout)),))
    ax, ad = A(x), A(d)
    ck(lib.mplbws_conv3x3_wgrad(ax.p, ad.p, dw.p, db.p, k.p, n, h, wd, cin, cout))
    ref, refb = nno.conv3x3_wgrad(x, d)
    mag, magb = nno.conv3x3_wgrad(np.abs(x), np.abs(d))
    # FP32 sums over the pixels
    m = n * h * wd
    assert (np.abs(dw.numpy() - ref) <= m * 2.0 ** -24 * mag).all()
    assert (np.abs(db.numpy() - refb) <= m * 2.0 ** -24 * magb + 1e-30).all()


def test_weight_gradient_drops_the_next_pixels_channels():
    """With channel counts that are no multiple of four the loads are wider than
    what is left of a pixel.  What they bring of another pixel is no part of a
    sum, even where it is no number: here that pixel is behind the array, which
    the rest of the allocation follows."""
    lib, rng = ws.load(), np.random.default_rng(14)
    n, h, wd, cin, cout = 1, 6, 21, 3, 5
    x = rng.standard_normal((n, h, wd, cin)).astype(np.float32)
    d = rng.standard_normal((n, h, wd, cout)).astype(np.float32)
    nan = np.full(64, np.nan, np.float32)
    ax = ws.DeviceArray.from_numpy(np.concatenate([nan, x.ravel(), nan]))
    ad = ws.DeviceArray.from_numpy(np.concatenate([nan, d.ravel(), nan]))
    dw, db = ws.DeviceArray((9, cin, cout)), ws.DeviceArray((cout,))
    k = ws.DeviceArray((int(lib.mplbws_wgrad_workspace(n, h, wd, cin, cout)),))
    ck(lib.mplbws_conv3x3_wgrad(at(ax, 64), at(ad, 64), dw.p, db.p, k.p, n, h, wd, cin, cout))
    ref, _ = nno.conv3x3_wgrad(x, d)
    mag, _ = nno.conv3x3_wgrad(np.abs(x), np.abs(d))
    assert (np.abs(dw.numpy() - ref) <= n * h * wd * 2.0 ** -24 * mag).all()
    assert np.isfinite(db.numpy()).all()


def _patches(lib, d, width, channels, starts, rng):
    """A zeroed array of `width` pixels with 40 random ones from each start on."""
    ck(lib.mplbws_zero(d.p, 4 * d.numel()))
    out = []
    for s in starts:
        a = rng.standard_normal((1, 1, 40, channels)).astype(np.float32)
        ck(lib.mplbws_upload(at(d, s * channels), a.ctypes.data, a.nbytes))
        out.append(a)
    return out


def test_convolution_of_rows_past_four_gib():
    """One row of 2^20 pixels x 1040 channels (4.4 GB), zero but for a few
    patches, one of them past the 32-bit offsets and at the row's end."""
    lib, rng = ws.load(), np.random.default_rng(15)
    wd, cin, cout = 1 << 20, 1040, 5
    starts = (0, 500001, wd - 40)
    assert (wd - 40) * cin * 4 > 1 << 32
    x, out = ws.DeviceArray((wd, cin)), ws.DeviceArray((wd, cout))
    patches = _patches(lib, x, wd, cin, starts, rng)
    w = (rng.standard_normal((9, cin, cout)) / 8).astype(np.float32)
    dw = ws.DeviceArray.from_numpy(w)
    ck(lib.mplbws_conv3x3_fwd(x.p, dw.p, None, out.p, 1, 1, wd, cin, cout, 0))
    got = out.numpy()
    for s, a in zip(starts, patches):
        mag = (9 * cin + 1) * 2.0 ** -24 * nno.conv3x3(np.abs(a), np.abs(w))[0, 0]
        assert (np.abs(got[s:s + 40] - nno.conv3x3(a, w)[0, 0]) <= mag).all(), s
    assert not got[41:500000].any() and not got[500042:wd - 41].any()


def test_convolution_of_weights_past_four_gib():
    lib, rng = ws.load(), np.random.default_rng(16)
    cin, cout = 10928, 10930
    assert 9 * cin * cout * 4 > 1 << 32
    x = rng.standard_normal((1, 1, 2, cin)).astype(np.float32)
    w = np.resize(rng.standard_normal(1000003).astype(np.float32), (9, cin, cout))
    dx, dw, out = ws.DeviceArray.from_numpy(x), ws.DeviceArray.from_numpy(w), ws.DeviceArray((2, cout))
    ck(lib.mplbws_conv3x3_fwd(dx.p, dw.p, None, out.p, 1, 1, 2, cin, cout, 0))
    some = np.r_[0:3, 5000:5003, cout - 3:cout]
    ws_ = np.ascontiguousarray(w[:, :, some])
    tol = (9 * cin + 1) * 2.0 ** -24 * nno.conv3x3(np.abs(x), np.abs(ws_))[0, 0]
    assert (np.abs(out.numpy()[:, some] - nno.conv3x3(x, ws_)[0, 0]) <= tol).all()


def test_weight_gradient_of_rows_past_four_gib():
    lib, rng = ws.load(), np.random.default_rng(17)
    wd, cin, cout = 1 << 20, 3, 1040
    starts = (0, 500001, wd - 40)
    x, d = ws.DeviceArray((wd, cin)), ws.DeviceArray((wd, cout))
    xs, ds = (_patches(lib, a, wd, c, starts, rng) for a, c in ((x, cin), (d, cout)))
    dw, db = ws.DeviceArray((9, cin, cout)), ws.DeviceArray((cout,))
    k = ws.DeviceArray((int(lib.mplbws_wgrad_workspace(1, 1, wd, cin, cout)),))
    ck(lib.mplbws_conv3x3_wgrad(x.p, d.p, dw.p, db.p, k.p, 1, 1, wd, cin, cout))
    ref, refb, mag, magb = 0, 0, 0, 0
    for a, b in zip(xs, ds):
        r, rb = nno.conv3x3_wgrad(a, b)
        m, mb = nno.conv3x3_wgrad(np.abs(a), np.abs(b))
        ref, refb, mag, magb = ref + r, refb + rb, mag + m, magb + mb
    # FP32 sums of 120 terms that are not zero
    assert (np.abs(dw.numpy() - ref) <= 120 * 2.0 ** -24 * mag).all()
    assert (np.abs(db.numpy() - refb) <= 120 * 2.0 ** -24 * magb + 1e-30).all()
