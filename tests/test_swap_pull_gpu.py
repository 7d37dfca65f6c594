"""The swap scheme in one pass per step (blocks of walls without connections)
against the CPU oracle, bit for bit: odd and even runs (the state returns to
one buffer), a graph replay, tile edges, every wall moving in another order,
several blocks, and a run restarted from its own f."""
import sys

import numpy as np
import pytest

from mplb_amd import cases, hip
from mplb_amd.enums import BoundaryScheme as BSch
from mplb_amd.enums import BoundarySurface as BS
from mplb_amd.enums import VertexType as VT
from oracle.oracle import OracleCase

pytestmark = pytest.mark.gpu


def log(m):
    print(m, flush=True)
    sys.stdout.flush()


def same(g, o, what):
    for b in g.sizes:
        assert np.array_equal(g.get_f(b), o.get_f(b)), (what, b)
    g.update_macros()
    o.update_macros()
    for b in g.sizes:
        for v in range(4):
            assert np.array_equal(g.get_macro(b, v), o.get_macro(b, v)), (what, b, v)


@pytest.mark.parametrize("size", [(3, 3, 3), (64, 5, 4), (66, 4, 7), (31, 19, 6), (16, 23, 3)])
def test_swap_pull_bitexact(size):
    log("swap pull %s" % (size,))
    g, o = hip.LatticeCase(3), OracleCase(3)
    for be in (g, o):
        cases.cavity3d_swap(be, max(size), re=90.0, noise=True, size=size)
    for n in (1, 2, 3, 37):
        g.step(n)
        o.step(n)
        same(g, o, n)
    f = g.get_f(0)
    for be in (g, o):
        be.set_f(0, f)
        be.step(5)
    same(g, o, "restart")
    g.close()


def test_swap_pull_large():
    """A lattice past the cache's size, against the oracle over a few steps."""
    log("swap pull 131 x 128 x 126")
    g, o = hip.LatticeCase(3), OracleCase(3)
    for be in (g, o):
        cases.cavity3d_swap(be, 131, re=90.0, noise=True, size=(131, 128, 126))
    g.step(3)
    o.step(3)
    assert np.array_equal(g.get_f(0), o.get_f(0))
    g.close()


@pytest.mark.parametrize("force", [None, (1e-4, -2e-4, 5e-5)])
def test_swap_pull_blocks_and_moving_walls(force):
    log("swap pull two blocks, moving walls, force %s" % (force,))
    sizes = [(17, 9, 11), (21, 6, 8)]

    def build(be):
        for b, n in enumerate(sizes):
            be.add_block(b, n)
        be.set_scheme(cases.SCHEME_SWAP)
        be.set_collision(cases.tau_ref_for(0.7, 1.0), force_type=1 if force else 0,
                         force_macros=bool(force))
        for b in range(2):
            for k, s in enumerate(("Front", "Left", "Top", "Back", "Right", "Bottom")):
                v = (0.01 * k, 0.02, -0.01 * k)
                be.add_boundary(b, BS[s], BSch.EQMDiffuseRefl, v, VT.Wall)
        be.prepare()
        for b, n in enumerate(sizes):
            if force:
                be.set_accel(b, force)
            shp = tuple(reversed(n))
            z = np.zeros(shp)
            be.set_macros(b, cases.density_noise(shp, amplitude=1e-3), z, z, z)
        be.init_feq()
        be.set_dt(1.0)

    g, o = hip.LatticeCase(3), OracleCase(3)
    build(g)
    build(o)
    g.step(40)
    o.step(40)
    same(g, o, "blocks")
    g.close()
