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


@pytest.mark.parametrize("name", ["pair", "tile", "march", "single", "swap", "channel"])
def test_timed_steps_are_those_of_step_f64(name, monkeypatch):
    """Bit for bit the oracle's state, in the launches of the form: only "single"
    has boundary kernels (the others end in a small case's one launch)."""
    monkeypatch.delenv("MPLBHIP_PAIR", raising=False)
    if name in ("march", "single"):
        monkeypatch.setenv("MPLBHIP_PAIR", "2" if name == "march" else "0")
        if name == "single":
            monkeypatch.setenv("MPLBHIP_FUSED", "0")
    build = {"pair": lambda be: cases.cavity3d(be, 44, re=100.0, size=(44, 41, 37)),
             "swap": lambda be: cases.cavity3d_swap(be, 20, size=(20, 13, 11)),
             "channel": lambda be: cases.channel2d(be, 40, 20, 0.8, 1e-5)}.get(
                 name, lambda be: cases.cavity2d(be, 40))
    dim = 3 if name in ("pair", "swap") else 2
    g, o = hip.LatticeCase(dim), OracleCase(dim)
    for be in (g, o):
        build(be)
    print("%s: %s" % (name, g.step_form()), flush=True)
    assert g.step_form()[0] == {"channel": "tile"}.get(name, name)
    for n in (1, 2, 3, 21, 40):
        total, kernels = g.step_timed(n)
        bulk, boundary = g.kernel_times()
        assert 0.0 < kernels <= total and kernels == pytest.approx(bulk + boundary)
        assert bulk > 0.0 and (boundary > 0.0) == (name == "single")
        g.step(n)
        o.step(2 * n)
        assert np.array_equal(g.get_f(0), o.get_f(0)), n
    g.close()
