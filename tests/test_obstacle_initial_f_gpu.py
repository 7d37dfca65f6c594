"""f before the first step is zero at obstacle nodes, as after it, whatever an
earlier read left in the buffer it is formed in."""
import numpy as np
import pytest

from mplb_amd import cases, hip
from oracle.oracle import OracleCase

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("storage", [hip.STORE_F64, hip.STORE_F32])
def test_initial_f_at_obstacles(storage):
    print("storage %d" % storage, flush=True)
    g, o = hip.LatticeCase(2, storage=storage), OracleCase(2)
    solid = cases.cavity2d_obstacles(g, 24, [(5, 5, 4, 3)])["solid"].astype(bool)
    cases.cavity2d_obstacles(o, 24, [(5, 5, 4, 3)])
    f0 = o.get_f(0)
    assert not f0[:, solid].any()
    g.set_f(0, f0 + 1.0)  # everywhere, and so in the buffer of the next read
    assert np.array_equal(g.get_f(0), f0 + 1.0)
    # (reading f refreshed the macros)
    g.set_macros(0, np.ones((24, 24)), np.zeros((24, 24)), np.zeros((24, 24)))
    g.init_feq()
    assert np.array_equal(g.get_f(0)[:, solid], f0[:, solid])
    if storage == hip.STORE_F64:
        assert np.array_equal(g.get_f(0), f0)
    g.close()
