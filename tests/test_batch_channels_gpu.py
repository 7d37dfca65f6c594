"""Batches of force-driven periodic channels go on after instances froze: the
halo copies of a block that stopped an odd number of launches before the others
are those of its own latest state."""
import numpy as np
import pytest

from mplb_amd import cases, hip
from oracle.oracle import OracleCase

pytestmark = pytest.mark.gpu

ONE_A, ONE_B = ("channel", [33], 9, 0.9, 2e-5), ("channel", [40], 12, 0.8, 1e-5)
TWO_A, TWO_B = ("channel", [20, 18], 9, 0.9, 2e-5), ("channel", [20, 18], 12, 0.8, 1e-5)


# several steps per launch: a period of 10 is three launches; single steps: one
# launch per step; linked blocks: single steps and merged halo copies
@pytest.mark.parametrize("specs, period, pair", [((ONE_A, ONE_B), 10, None),
                                                 ((ONE_A, ONE_B), 25, "0"),
                                                 ((ONE_A, TWO_B), 25, None),
                                                 ((TWO_A, TWO_B), 5, None)])
def test_batch_of_channels_goes_on_after_freezing_f64(specs, period, pair, monkeypatch):
    print("channels %s period %d pair %s" % (specs, period, pair), flush=True)
    monkeypatch.delenv("MPLBHIP_PAIR", raising=False)
    if pair is not None:
        monkeypatch.setenv("MPLBHIP_PAIR", pair)
    g = hip.LatticeCase(2, storage=hip.STORE_F64, device=0)
    insts = cases.batched_mixed(g, specs)
    steps, _, done = g.iterate_batch(1e-4, period, 4000)
    print("steps %s done %d" % (list(steps), done), flush=True)
    assert np.all(steps > 0) and done == max(steps)
    first, last = (int(steps[i["blocks"][0]]) for i in insts)
    # an odd number of periods, each an odd number of launches
    assert last > first and (last - first) // period % 2 == 1
    oracles = []
    for inst, spec in zip(insts, specs):
        o = OracleCase(2)
        cases.channel_multi(o, *spec[1:])
        o.step(int(steps[inst["blocks"][0]]))
        oracles.append(o)

    def compare(what):
        for inst, o in zip(insts, oracles):
            for k, b in enumerate(inst["blocks"]):
                assert np.array_equal(g.get_f(b), o.get_f(k)), (what, b)

    compare("frozen")
    g.step(17)
    for o in oracles:
        o.step(17)
    compare("stepped")
    # (no residual is below zero: every instance takes every step)
    g.iterate_batch(0.0, period, 23)
    for o in oracles:
        o.step(23)
    compare("iterated")
    g.close()
