"""mplbhip_step_timed takes the steps of mplbhip_step and none besides."""
import numpy as np
import pytest

from mplb_amd import cases, hip
from oracle.oracle import OracleCase

pytestmark = pytest.mark.gpu


def test_no_timed_steps_leave_a_large_case_as_it_is():
    """From 2^20 nodes on the single-step launch is tuned by dry steps, which
    need a real one after them."""
    g = hip.LatticeCase(3, storage=hip.STORE_F32)
    cases.cavity3d(g, 104, re=100.0, size=(104, 103, 102))
    g.step(10)
    f, mass = g.get_f(0), g.mass()
    print("step_timed(0) after 10 steps", flush=True)
    assert g.step_timed(0) == (pytest.approx(0.0, abs=5.0), 0.0)
    assert np.array_equal(g.get_f(0), f) and g.mass() == mass
    g.update_macros()
    rho = g.get_macro(0, 0)
    g.step_timed(0)
    g.update_macros()
    assert np.array_equal(g.get_macro(0, 0), rho)
    g.close()


def test_timed_swap_steps_keep_the_launch_shape_f64():
    """The swap scheme has no single-step launch to tune."""
    size = (104, 103, 102)
    g, o = hip.LatticeCase(3), OracleCase(3)
    for be in (g, o):
        cases.cavity3d_swap(be, 104, size=size)
    shape = g.launch_shape()
    print("swap %s shape %s" % (size, shape), flush=True)
    for n in (3, 0, 2):
        total, kernels = g.step_timed(n)
        assert (kernels > 0.0) == (n > 0)
        o.step(n)
        assert np.array_equal(g.get_f(0), o.get_f(0)), n
        assert g.launch_shape() == shape
    g.close()
