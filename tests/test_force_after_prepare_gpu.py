"""A body force given or taken away after mplbhip_prepare: the steps run in the
form that the case has from then on, tuned where that is single steps."""
import numpy as np
import pytest

from mplb_amd import cases, hip

pytestmark = pytest.mark.gpu


def build(be, size):
    dim, dt = len(size), 0.01
    tau = cases.tau_ref_for(0.7, dt)
    if dim == 3:
        cases.cavity3d(be, max(size), re=100.0, size=size)
        return cases.tau_ref_for(cases.cavity_params(max(size), 100.0, 0.05)[2],
                                 cases.cavity_params(max(size), 100.0, 0.05)[1])
    cases.cavity2d(be, size[0], rho0=cases.density_noise(size[::-1]))
    return tau


@pytest.mark.parametrize("n, storage", [(1100, hip.STORE_F64), (1100, hip.STORE_F32), (90, hip.STORE_F64)])
def test_force_after_prepare_2d(n, storage, monkeypatch):
    out = []
    for pair in (None, "0"):
        monkeypatch.delenv("MPLBHIP_PAIR", raising=False)
        if pair:
            monkeypatch.setenv("MPLBHIP_PAIR", pair)
        g = hip.LatticeCase(2, storage=storage)
        tau = build(g, (n, n))
        forms = [g.step_form()[0]]
        g.step(11)
        g.set_collision(tau, force_type=1, force_macros=True)
        g.set_accel(0, (1e-5, -2e-5))
        forms.append(g.step_form()[0])
        g.step(45)
        g.set_collision(tau)
        forms.append(g.step_form()[0])
        g.step(9)
        out.append(g.get_f(0))
        g.close()
        print("%d^2 storage %d pair %s: %s" % (n, storage, pair, forms), flush=True)
        if pair:
            assert forms == ["single"] * 3
        else:
            assert forms == (["march", "tile", "march"] if n > 1024 else ["tile"] * 3)
    if storage == hip.STORE_F64:
        assert np.array_equal(out[0], out[1])
    else:
        # a node's update and its wall round a few times each, of values of at
        # most 1/2: 8 half units in the last place of 1/2 per step
        assert np.abs(out[0] - out[1]).max() <= 65 * 8 * 2.0 ** -26


def test_force_after_the_first_steps_tunes_single_steps_3d(monkeypatch, capfd):
    monkeypatch.delenv("MPLBHIP_PAIR", raising=False)
    monkeypatch.setenv("MPLBHIP_VERBOSE", "1")
    size = (104, 103, 102)
    g = hip.LatticeCase(3, storage=hip.STORE_F32)
    tau = build(g, size)
    assert g.step_form() == ("pair", 2)
    g.step(10)
    assert "autotune picked" not in capfd.readouterr().err
    g.set_collision(tau, force_type=1, force_macros=True)
    g.set_accel(0, (1e-5, 0.0, 0.0))
    assert g.step_form() == ("single", 1)
    g.step(40)
    assert capfd.readouterr().err.count("autotune picked") == 1
    f = g.get_f(0)
    g.close()
    monkeypatch.setenv("MPLBHIP_PAIR", "0")
    r = hip.LatticeCase(3, storage=hip.STORE_F32)
    build(r, size)
    r.step(10)
    r.set_collision(tau, force_type=1, force_macros=True)
    r.set_accel(0, (1e-5, 0.0, 0.0))
    r.step(40)
    # (the same rounding node by node in every FP32 form of a plain cavity;
    # walls of the tuned fold levels may round a few times differently)
    assert np.abs(f - r.get_f(0)).max() <= 50 * 8 * 2.0 ** -26
    r.close()
