"""Several steps per launch of 2D blocks: in LDS tiles (the default form of
smaller cases and of x-periodic channels) and marching through the rows
(larger ones; MPLBHIP_PAIR=2 forces it), against the CPU oracle in FP64, bit
for bit, and against single steps in reduced storage, at tile and strip edges,
with remainders of every kind."""
import sys

import numpy as np
import pytest

from mplb_amd import cases, hip
from mplb_amd.enums import BoundaryScheme as BSch
from mplb_amd.enums import BoundarySurface as BS
from mplb_amd.enums import VertexType as VT
from oracle.oracle import OracleCase

pytestmark = pytest.mark.gpu

# one tile and its edges, several; (150, 131) has more tiles of 8 x 8 than the
# chip has CUs and runs in tiles of 16 x 16
TILE = [(3, 3), (8, 17), (16, 40), (33, 8), (120, 130), (150, 131)]
# one to four row groups per wave, a strip and its edges, several strips
MARCH = [(3, 3), (5, 70), (17, 33), (33, 40), (64, 9), (65, 16), (131, 17), (600, 31)]
FORMS = [("1", s) for s in TILE] + [("2", s) for s in MARCH]
RUNS = (1, 2, 3, 9, 40)  # alone, in one short launch, in several and a rest


def log(m):
    print(m, flush=True)
    sys.stdout.flush()


def cavity(be, size, lid=(cases.CS * 0.05, 0.0), order=("Left", "Right", "Top", "Bottom"),
           others=(0.0, 0.0)):
    dt, tau = cases.cavity_params(max(size), 100.0, 0.05)[1:]
    be.add_block(0, size)
    be.set_collision(cases.tau_ref_for(tau, dt))
    for s in order:
        be.add_boundary(0, BS[s], BSch.EQMDiffuseRefl, lid if s == "Top" else others, VT.Wall)
    be.prepare()
    shp = tuple(reversed(size))
    be.set_macros(0, cases.density_noise(shp), np.zeros(shp), np.zeros(shp))
    be.init_feq()
    be.set_dt(dt)


def same_as_oracle(build, runs=RUNS):
    g, o = hip.LatticeCase(2), OracleCase(2)
    build(g)
    build(o)
    for n in runs:
        g.step(n)
        o.step(n)
        assert np.array_equal(g.get_f(0), o.get_f(0)), n
    g.update_macros()
    o.update_macros()
    for v in range(3):
        assert np.array_equal(g.get_macro(0, v), o.get_macro(0, v)), v
    g.close()


def same_as_single_steps(build, storage, form, monkeypatch, n=41):
    out = []
    for pair in (form, "0"):
        monkeypatch.setenv("MPLBHIP_PAIR", pair)
        g = hip.LatticeCase(2, storage=storage)
        build(g)
        g.step(n)
        out.append(g.get_f(0))
        g.close()
    if storage == hip.STORE_F64:
        assert np.array_equal(out[0], out[1])
    elif storage == hip.STORE_F32:
        # a node's update and its wall round a few times each, of values of
        # at most 1/2: 8 half units in the last place of 1/2 per step
        assert np.abs(out[0] - out[1]).max() <= n * 8 * 2.0 ** -26
    else:
        # half has 11 bits: a population's rounding is below 2^-11 of the
        # largest deviation it reaches, at most once per step
        big = np.abs(out[1] - out[1].mean(axis=(1, 2), keepdims=True)).max()
        assert np.abs(out[0] - out[1]).max() <= n * 2.0 ** -11 * max(big, 1e-3)


@pytest.mark.parametrize("form,size", FORMS)
def test_steps2d_f64_bitexact(form, size, monkeypatch):
    log("steps2d F64 %s %s" % (form, size))
    monkeypatch.setenv("MPLBHIP_PAIR", form)
    same_as_oracle(lambda be: cavity(be, size))


@pytest.mark.parametrize("storage", [hip.STORE_F32, hip.STORE_F16])
@pytest.mark.parametrize("form,size", FORMS)
def test_steps2d_reduced_storage(form, size, storage, monkeypatch):
    log("steps2d storage %d %s %s" % (storage, form, size))
    same_as_single_steps(lambda be: cavity(be, size), storage, form, monkeypatch)


@pytest.mark.parametrize("storage", [hip.STORE_F64, hip.STORE_F32, hip.STORE_F16])
def test_steps2d_large_tiles(storage, monkeypatch):
    log("steps2d large tiles %d" % storage)
    same_as_single_steps(lambda be: cavity(be, (530, 497)), storage, "1", monkeypatch)


@pytest.mark.parametrize("form", ["1", "2"])
def test_steps2d_moving_walls_f64(form, monkeypatch):
    """Every wall moving, the faces defined in another order: the last-defined
    wall owns the corners."""
    monkeypatch.setenv("MPLBHIP_PAIR", form)
    same_as_oracle(lambda be: cavity(be, (37, 25), (0.05, 0.02), ("Top", "Right", "Bottom", "Left"),
                                     (0.01, 0.03)))


@pytest.mark.parametrize("size", [(32, 3), (41, 20), (48, 33), (301, 127)])
def test_steps2d_channel_f64(size, monkeypatch):
    """Tiles that wrap along x, with a body force; single steps after them
    read the halos that they left out."""
    log("steps2d channel %s" % (size,))
    monkeypatch.setenv("MPLBHIP_PAIR", "1")
    same_as_oracle(lambda be: cases.channel2d(be, size[0], size[1], 0.8, 1e-5), RUNS + (1, 17))


@pytest.mark.parametrize("size", [(7, 30), (61, 44), (1040, 1020)])
def test_steps2d_forced_cavity_f64(size, monkeypatch):
    """A body force between four walls: tiles at every size."""
    log("steps2d forced cavity %s" % (size,))

    def build(be):
        be.add_block(0, size)
        be.set_collision(cases.tau_ref_for(0.8, 1.0), force_type=1, force_macros=True)
        for s in ("Left", "Right", "Top", "Bottom"):
            be.add_boundary(0, BS[s], BSch.EQMDiffuseRefl, (0.0, 0.01), VT.Wall)
        be.prepare()
        be.set_accel(0, (1e-5, -2e-5))
        shp = tuple(reversed(size))
        be.set_macros(0, cases.density_noise(shp), np.zeros(shp), np.zeros(shp))
        be.init_feq()
        be.set_dt(1.0)

    same_as_oracle(build, RUNS if size[0] < 1000 else (6,))


@pytest.mark.parametrize("storage", [hip.STORE_F32, hip.STORE_F16])
def test_steps2d_channel_reduced_storage(storage, monkeypatch):
    same_as_single_steps(lambda be: cases.channel2d(be, 101, 60, 0.8, 1e-5), storage, "1",
                         monkeypatch)


@pytest.mark.parametrize("storage", [hip.STORE_F64, hip.STORE_F32, hip.STORE_F16])
@pytest.mark.parametrize("form", ["1", "2"])
@pytest.mark.parametrize("n", [24, 131])
def test_steps2d_obstacles(n, form, storage, monkeypatch):
    log("steps2d obstacles %d %s %d" % (n, form, storage))
    rects = [(4, 5, 6, 3), (n // 2, n // 3, 5, 7)]
    same_as_single_steps(lambda be: cases.cavity2d_obstacles(be, n, rects), storage, form,
                         monkeypatch)


@pytest.mark.parametrize("form", ["1", "2"])
def test_steps2d_graph_replays_f64(form, monkeypatch):
    """Runs of whole graphs of 16 launches, with and without a rest, and the
    single steps after them; the periodic channel's halos too."""
    monkeypatch.setenv("MPLBHIP_PAIR", form)
    same_as_oracle(lambda be: cavity(be, (70, 19)), (300, 129, 1, 131))
    if form == "1":
        same_as_oracle(lambda be: cases.channel2d(be, 45, 18, 0.8, 1e-5), (257, 2, 140))


@pytest.mark.parametrize("form", ["1", "2"])
def test_steps2d_iterate_and_restart_f64(form, monkeypatch):
    """Check steps after launches of several steps, a residual, and a run
    restarted from its own f."""
    monkeypatch.setenv("MPLBHIP_PAIR", form)
    g, o = hip.LatticeCase(2), OracleCase(2)
    cavity(g, (70, 19))
    cavity(o, (70, 19))
    done, res = g.iterate(0.0, 9, 33)
    assert done == 33
    o.step(27)
    o.update_macros()
    o.step(6)
    f = g.get_f(0)
    assert np.array_equal(f, o.get_f(0))
    g.set_f(0, f)
    o.set_f(0, f)
    g.step(10)
    o.step(10)
    assert np.array_equal(g.get_f(0), o.get_f(0))
    g.close()


@pytest.mark.parametrize("form", ["1", "2"])
def test_steps2d_batch_of_blocks_freezes_f64(form, monkeypatch):
    """Blocks of different sizes: each stops at its own convergence and keeps
    its state, the others go on."""
    monkeypatch.setenv("MPLBHIP_PAIR", form)
    sizes, res = [24, 33, 16], [40.0, 100.0, 20.0]
    g = hip.LatticeCase(2)
    cases.batched_cavities(g, sizes, res)
    steps, resid, done = g.iterate_batch(2e-3, 25, 4000)
    log("steps %s" % list(steps))
    assert (steps > 0).all() and len(set(steps)) > 1
    for b, (n, re) in enumerate(zip(sizes, res)):
        monkeypatch.setenv("MPLBHIP_PAIR", "0")
        s = hip.LatticeCase(2)
        cases.batched_cavities(s, [n], [re])
        s.step(int(steps[b]))
        assert np.array_equal(g.get_f(b), s.get_f(0)), b
        s.close()
    g.close()
