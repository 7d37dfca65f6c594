"""The warm-start network's layers at the edges of their kernels' tiles and
vector widths: upsampling and channel copies exactly, convolutions against the
CPU layer oracle (BF16 operands, float64 sums)."""
import sys

import numpy as np
import pytest

from mplb_amd import warmstart as ws
from oracle import nn_oracle as nno

pytestmark = pytest.mark.gpu


def log(m):
    print(m, flush=True)
    sys.stdout.flush()


def ck(rc):
    assert rc == 0, rc


# channel counts and offsets of four-float accesses, and of none
@pytest.mark.parametrize("c,ctot,c0", [(8, 8, 0), (4, 20, 8), (12, 17, 4), (3, 9, 5), (6, 8, 2)])
@pytest.mark.parametrize("n,h,wd", [(1, 1, 1), (3, 5, 7), (2, 9, 130)])
def test_upsampling_and_channel_copies(n, h, wd, c, ctot, c0):
    log("up and channels %s" % ((n, h, wd, c, ctot, c0),))
    lib, rng = ws.load(), np.random.default_rng(5)
    A = ws.DeviceArray.from_numpy
    x = rng.standard_normal((n, h, wd, c)).astype(np.float32)
    wide = rng.standard_normal((n, 2 * h, 2 * wd, ctot)).astype(np.float32)
    dx, dw = A(x), A(wide)
    ck(lib.mplbws_up2_fwd(dx.p, dw.p, n, h, wd, c, ctot, c0))
    ref = wide.copy()
    ref[..., c0:c0 + c] = x.repeat(2, axis=1).repeat(2, axis=2)
    assert np.array_equal(dw.numpy(), ref)
    fine = rng.standard_normal(wide.shape).astype(np.float32)
    df = A(fine)
    ck(lib.mplbws_up2_bwd(df.p, dx.p, n, h, wd, c, ctot, c0))
    f = fine[..., c0:c0 + c]
    assert np.array_equal(dx.numpy(), (f[:, ::2, ::2] + f[:, ::2, 1::2])
                          + (f[:, 1::2, ::2] + f[:, 1::2, 1::2]))
    thin = rng.standard_normal((n, 2 * h, 2 * wd, c)).astype(np.float32)
    dt, pixels = A(thin), n * 4 * h * wd
    ck(lib.mplbws_channels(df.p, dt.p, pixels, c, ctot, c0, 2))
    assert np.array_equal(dt.numpy(), thin + f)
    ck(lib.mplbws_channels(df.p, dt.p, pixels, c, ctot, c0, 1))
    assert np.array_equal(dt.numpy(), f)
    dt = A(thin)
    ck(lib.mplbws_channels(dt.p, df.p, pixels, c, ctot, c0, 0))
    ref = fine.copy()
    ref[..., c0:c0 + c] = thin
    assert np.array_equal(df.numpy(), ref)


# (n, h, w, cin, cout): one pixel, tiles of 32 columns and their edges, rows
# past a tile, chunks of 32 input channels with remainders of 8 and 16, 4-, 1-
# and 3-channel remainders of the output, the larger tiles' smallest grid
CONV = [(1, 1, 1, 8, 4), (2, 3, 2, 8, 1), (1, 5, 33, 24, 24), (3, 32, 32, 40, 36),
        (1, 17, 65, 48, 33), (2, 40, 31, 72, 64), (1, 9, 100, 56, 67), (33, 64, 64, 8, 8),
        (1, 70, 7, 16, 32)]


@pytest.mark.parametrize("n,h,wd,cin,cout", CONV)
def test_convolution_forward(n, h, wd, cin, cout):
    log("conv %s" % ((n, h, wd, cin, cout),))
    lib, rng = ws.load(), np.random.default_rng(7)
    A = ws.DeviceArray.from_numpy
    x = rng.standard_normal((n, h, wd, cin)).astype(np.float32)
    w = (rng.standard_normal((9, cin, cout)) / 8).astype(np.float32)
    b = rng.standard_normal(cout).astype(np.float32)
    dx, dw, db, out = A(x), A(w), A(b), ws.DeviceArray((n, h, wd, cout))
    mag = nno.conv3x3(np.abs(x), np.abs(w)) + np.abs(b)
    for bias, relu in ((True, 1), (False, 0)):
        ck(lib.mplbws_conv3x3_fwd(dx.p, dw.p, db.p if bias else None, out.p, n, h, wd, cin, cout,
                                  relu))
        ref = nno.conv3x3(x, w, b if bias else None, relu=bool(relu))
        # FP32 sums of 9 cin exact products and the bias: at most that many
        # roundings of partial sums bounded by the sum of magnitudes
        tol = (9 * cin + 1) * 2.0 ** -24 * mag
        assert (np.abs(out.numpy() - ref) <= tol).all()


# sub-tiles of 16 to 64 columns and their remainders, several segments of a
# row, several chunks of an image (64 x 100 rows of 41), channels of one, two
# and three tiles of 32 with remainders that are no multiple of 4
@pytest.mark.parametrize("n,h,wd,cin,cout",
                         [(1, 1, 1, 8, 4), (3, 2, 17, 5, 3), (2, 16, 16, 32, 32),
                          (1, 33, 48, 40, 36), (2, 21, 65, 72, 24), (1, 9, 130, 8, 67),
                          (2, 100, 64, 33, 12)])
def test_convolution_weight_gradient(n, h, wd, cin, cout):
    log("wgrad %s" % ((n, h, wd, cin, cout),))
    lib, rng = ws.load(), np.random.default_rng(9)
    A = ws.DeviceArray.from_numpy
    x = rng.standard_normal((n, h, wd, cin)).astype(np.float32)
    d = rng.standard_normal((n, h, wd, cout)).astype(np.float32)
    dw, db = ws.DeviceArray((9, cin, cout)), ws.DeviceArray((cout,))
    k = ws.DeviceArray((int(lib.mplbws_wgrad_workspace(n, h, wd, cin, cout)),))
    ax, ad = A(x), A(d)
    ck(lib.mplbws_conv3x3_wgrad(ax.p, ad.p, dw.p, db.p, k.p, n, h, wd, cin, cout))
    ref, refb = nno.conv3x3_wgrad(x, d)
    mag, magb = nno.conv3x3_wgrad(np.abs(x), np.abs(d))
    # FP32 sums over the pixels, as for the forward convolution
    m = n * h * wd
    assert (np.abs(dw.numpy() - ref) <= m * 2.0 ** -24 * mag).all()
    assert (np.abs(db.numpy() - refb) <= m * 2.0 ** -24 * magb + 1e-30).all()
    again = ws.DeviceArray((9, cin, cout))
    ck(lib.mplbws_conv3x3_wgrad(ax.p, ad.p, again.p, None, k.p, n, h, wd, cin, cout))
    assert np.array_equal(again.numpy(), dw.numpy())
