"""Two steps per launch (the default form of 3D cavities from 2^16 nodes on;
MPLBHIP_PAIR=1 forces it): against the CPU oracle in FP64, bit for bit, and
against the single-step forms in FP32 (bit for bit: the same roundings node by
node) and FP16 (the rounding of each wall node differs between the single-step
forms themselves), at tile edges, with remainders of every kind."""
import sys

import numpy as np
import pytest

from mplb_amd import cases, hip
from mplb_amd.enums import BoundaryScheme as BSch
from mplb_amd.enums import BoundarySurface as BS
from mplb_amd.enums import VertexType as VT
from oracle.oracle import OracleCase

pytestmark = pytest.mark.gpu

# rows of one node past a tile, below a tile, of several tiles; one tile's
# height and one node more; three planes (every plane a face's neighbour)
SIZES = [(16, 4, 3), (17, 11, 12), (33, 23, 9), (65, 40, 17), (130, 5, 9)]


def log(m):
    print(m, flush=True)
    sys.stdout.flush()


def cavity(be, size):
    return cases.cavity3d(be, max(size), re=100.0, noise=True, size=size)


@pytest.mark.parametrize("lattice", [19, 15])
@pytest.mark.parametrize("size", SIZES)
def test_pair_f64_bitexact(size, lattice, monkeypatch):
    log("pair F64 %s D3Q%d" % (size, lattice))
    monkeypatch.setenv("MPLBHIP_PAIR", "1")
    g = hip.LatticeCase(3, storage=hip.STORE_F64, lattice=lattice)
    o = OracleCase(3, lattice=lattice) if lattice == 15 else OracleCase(3)
    cavity(g, size)
    cavity(o, size)
    for n in (1, 2, 3, 40):  # odd and even runs, a graph replay
        g.step(n)
        o.step(n)
        assert np.array_equal(g.get_f(0), o.get_f(0)), n
    g.update_macros()
    o.update_macros()
    for v in range(4):
        assert np.array_equal(g.get_macro(0, v), o.get_macro(0, v)), v
    assert abs(g.mass() - o.mass()) <= 1e-13 * abs(o.mass())
    g.close()


@pytest.mark.parametrize("size", SIZES)
@pytest.mark.parametrize("storage", [hip.STORE_F32, hip.STORE_F16])
@pytest.mark.parametrize("lattice", [19, 15])
def test_pair_reduced_storage(size, storage, lattice, monkeypatch):
    log("pair storage %d %s D3Q%d" % (storage, size, lattice))
    out = []
    for pair in ("1", "0"):
        monkeypatch.setenv("MPLBHIP_PAIR", pair)
        g = hip.LatticeCase(3, storage=storage, lattice=lattice)
        cavity(g, size)
        g.step(41)
        out.append(g.get_f(0))
        g.close()
    if storage == hip.STORE_F32:
        assert np.array_equal(out[0], out[1])
    else:
        # half has 11 bits: a population's rounding is below 2^-11 of the
        # largest deviation it reaches, and 41 steps at tau > 1/2 add it up
        # at most once per step
        big = np.abs(out[1] - out[1].mean(axis=(1, 2, 3), keepdims=True)).max()
        assert np.abs(out[0] - out[1]).max() <= 41 * 2.0 ** -11 * max(big, 1e-3)


def test_pair_boundary_orders_and_moving_walls_f64(monkeypatch):
    """Every wall moving and the faces defined in another order: the
    last-defined wall owns the edges and corners."""
    monkeypatch.setenv("MPLBHIP_PAIR", "1")
    size = (37, 25, 14)

    def build(be):
        be.add_block(0, size)
        dt = 1.0 / 36 / cases.CS
        be.set_collision(cases.tau_ref_for(0.7, dt))
        vel = {"Front": (0.02, 0.01, 0.0), "Left": (0.0, 0.03, -0.01), "Top": (0.05, 0.0, 0.02),
               "Back": (0.0, 0.0, 0.0), "Right": (0.0, -0.02, 0.03), "Bottom": (0.01, 0.0, 0.01)}
        for s in ("Front", "Left", "Top", "Back", "Right", "Bottom"):
            be.add_boundary(0, BS[s], BSch.EQMDiffuseRefl, vel[s], VT.Wall)
        be.prepare()
        shp = tuple(reversed(size))
        z = np.zeros(shp)
        be.set_macros(0, cases.density_noise(shp), z, z, z)
        be.init_feq()
        be.set_dt(dt)

    g, o = hip.LatticeCase(3), OracleCase(3)
    build(g)
    build(o)
    for n in (7, 30):
        g.step(n)
        o.step(n)
        assert np.array_equal(g.get_f(0), o.get_f(0)), n
    g.close()


def test_pair_iterate_and_restart_f64(monkeypatch):
    """Check steps between two-step launches, a residual, and a run restarted
    from its own f."""
    monkeypatch.setenv("MPLBHIP_PAIR", "1")
    size = (34, 19, 21)
    g, o = hip.LatticeCase(3), OracleCase(3)
    cavity(g, size)
    cavity(o, size)
    done, res = g.iterate(0.0, 7, 29)
    assert done == 29
    o.step(28)
    o.update_macros()
    for v in range(4):
        assert np.array_equal(g.get_macro(0, v), o.get_macro(0, v)), v
    o.step(1)
    f = g.get_f(0)
    assert np.array_equal(f, o.get_f(0))
    g.set_f(0, f)
    o.set_f(0, f)
    g.step(10)
    o.step(10)
    assert np.array_equal(g.get_f(0), o.get_f(0))
    g.close()


def test_pair_batch_of_blocks_freezes_f64(monkeypatch):
    """Unconnected 3D blocks of different sizes: each stops at its own
    convergence and keeps its state, the others go on."""
    monkeypatch.setenv("MPLBHIP_PAIR", "1")
    sizes, res = [(18, 12, 9), (33, 16, 16), (20, 20, 20)], [5.0, 20.0, 60.0]
    dts = []

    def block(be, b, size, re, own):
        mesh, dt, tau_l = cases.cavity_params(max(size), re, 0.05)
        be.add_block(b, size)
        for s in ("Left", "Right", "Top", "Bottom", "Front", "Back"):
            v = (cases.CS * 0.05, 0.0, 0.0) if s == "Top" else (0.0, 0.0, 0.0)
            be.add_boundary(b, BS[s], BSch.EQMDiffuseRefl, v, VT.Wall)
        if not own:
            be.set_block_collision(b, cases.tau_ref_for(tau_l, dt), dt)
        return cases.tau_ref_for(tau_l, dt), dt

    g = hip.LatticeCase(3)
    for b, (n, re) in enumerate(zip(sizes, res)):
        dts.append(block(g, b, n, re, False))
    g.set_collision(1.0)
    g.prepare()
    for b, n in enumerate(sizes):
        shp = tuple(reversed(n))
        z = np.zeros(shp)
        g.set_macros(b, np.ones(shp), z, z, z)
    g.init_feq()
    steps, resid, done = g.iterate_batch(2e-3, 25, 4000)
    log("steps %s" % list(steps))
    assert (steps > 0).all() and len(set(steps)) > 1
    for b, (n, re) in enumerate(zip(sizes, res)):
        o = OracleCase(3)
        tau, dt = block(o, 0, n, re, True)
        o.set_collision(tau)
        o.prepare()
        shp = tuple(reversed(n))
        z = np.zeros(shp)
        o.set_macros(0, np.ones(shp), z, z, z)
        o.init_feq()
        o.set_dt(dt)
        o.step(int(steps[b]))
        assert np.array_equal(g.get_f(b), o.get_f(0)), b
    g.close()
