"""The warm-start network's layers at the edges of their kernels' tiles and
vector widths: upsampling and channel copies exactly."""
import sys

import numpy as np
import pytest

from mplb_amd import warmstart as ws

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
