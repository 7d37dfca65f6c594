"""Which kernel form a case's steps run in (mplbhip_step_form): the cases that
the tests of each form build, by size and as MPLBHIP_PAIR forces them, and cases
that no form of several steps takes."""
import numpy as np
import pytest

from mplb_amd import cases, hip
from mplb_amd.enums import BoundaryScheme as BSch
from mplb_amd.enums import BoundarySurface as BS
from mplb_amd.enums import VertexType as VT
from tests import test_pair_gpu, test_steps2d_gpu

pytestmark = pytest.mark.gpu

F64, F32, F16 = hip.STORE_F64, hip.STORE_F32, hip.STORE_F16


@pytest.fixture(autouse=True)
def environment(monkeypatch):
    for name in ("PAIR", "FUSED", "XFACE_FOLD", "XGROUP", "H2", "XCD_REMAP"):
        monkeypatch.delenv("MPLBHIP_" + name, raising=False)


def form(dim, build, storage=F64, lattice=None):
    g = hip.LatticeCase(dim, storage=storage, lattice=lattice)
    build(g)
    out = g.step_form()
    g.close()
    print("%s storage %d" % (out, storage), flush=True)
    return out


def obstacles(be):
    cases.cavity2d_obstacles(be, 24, [(5, 5, 4, 3)])


def outlet3(be):
    """A cavity with a pressure outlet."""
    size = (40, 40, 41)
    be.add_block(0, size)
    be.set_collision(cases.tau_ref_for(0.8, 0.01))
    for s in ("Left", "Right", "Top", "Bottom", "Front"):
        be.add_boundary(0, BS[s], BSch.EQMDiffuseRefl, (0.0, 0.0, 0.0), VT.Wall)
    be.add_boundary(0, BS.Back, BSch.ExtrapolPressure1ST, (1.0,), VT.OutLet)
    be.prepare()


@pytest.mark.parametrize("storage", [F64, F32, F16])
def test_forms_that_the_environment_asks_for(storage, monkeypatch):
    monkeypatch.setenv("MPLBHIP_PAIR", "1")
    for lattice in (19, 15):
        for size in test_pair_gpu.SIZES:
            assert form(3, lambda be: test_pair_gpu.cavity(be, size), storage,
                        lattice) == ("pair", 2), (size, lattice)
    for pair, size in test_steps2d_gpu.FORMS:
        monkeypatch.setenv("MPLBHIP_PAIR", pair)
        name, steps = form(2, lambda be: test_steps2d_gpu.cavity(be, size), storage)
        assert name == ("tile" if pair == "1" else "march") and steps > 2, size
    for pair, name in (("1", "tile"), ("2", "march")):
        monkeypatch.setenv("MPLBHIP_PAIR", pair)
        assert form(2, obstacles, storage)[0] == name
    monkeypatch.setenv("MPLBHIP_PAIR", "0")
    assert form(3, lambda be: cases.cavity3d(be, 48), storage) == ("single", 1)
    assert form(2, lambda be: cases.cavity2d(be, 48), storage) == ("single", 1)


@pytest.mark.parametrize("storage", [F64, F32, F16])
def test_forms_by_size(storage):
    assert form(3, lambda be: cases.cavity3d(be, 40), storage) == ("single", 1)
    assert form(3, lambda be: cases.cavity3d(be, 41), storage) == ("pair", 2)
    assert form(2, lambda be: cases.cavity2d(be, 128), storage) == ("tile", 8)
    assert form(2, lambda be: cases.cavity2d(be, 512), storage) == ("tile", 4)
    big = form(2, lambda be: cases.cavity2d(be, 1100), storage)
    assert big == ("march", {F64: 5, F32: 7, F16: 4}[storage])
    assert form(2, lambda be: cases.channel2d(be, 64, 20, 0.8, 1e-6), storage) == ("tile", 8)
    assert form(2, lambda be: cases.channel2d(be, 1200, 1000, 0.8, 1e-6), storage) == ("tile", 4)


def test_forms_of_the_swap_scheme():
    assert form(3, lambda be: cases.cavity3d_swap(be, 12)) == ("swap", 1)
    one = np.ones((5, 6, 7))
    assert form(3, lambda be: cases.swap_box(be, (7, 6, 5), 0.8, one, 0 * one, 0 * one,
                                             0 * one)) == ("single", 1)


def test_cases_of_single_steps(monkeypatch):
    """What the forms refuse, also where the environment asks for them."""
    monkeypatch.setenv("MPLBHIP_PAIR", "1")
    one = np.ones((40, 40, 40))
    # connections; rows too short for a tile; a boundary that is no wall
    assert form(3, lambda be: cases.periodic_box(be, (40, 40, 40), 0.8, one, 0 * one, 0 * one,
                                                 0 * one)) == ("single", 1)
    assert form(3, lambda be: cases.cavity3d(be, 15)) == ("single", 1)
    assert form(3, outlet3) == ("single", 1)
    assert form(2, lambda be: cases.channel2d(be, 31, 40, 0.8, 1e-6)) == ("single", 1)
    assert form(2, lambda be: cases.channel_multi(be, [40, 40], 9, 0.8, 1e-6)) == ("single", 1)
    # a single-step form chosen by the environment is the one that runs
    monkeypatch.delenv("MPLBHIP_PAIR")
    monkeypatch.setenv("MPLBHIP_XFACE_FOLD", "1")
    assert form(3, lambda be: cases.cavity3d(be, 48)) == ("single", 1)
