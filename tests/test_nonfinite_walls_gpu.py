"""What is not a number spreads as in the reference's loops: a wall reads its
incoming populations only, so a wall node whose neighbour along the wall has
none stays finite.  In every form of the step, against the CPU oracle: FP64 bit
for bit, reduced storage by the nodes that are reached."""
import numpy as np
import pytest

from mplb_amd import cases, hip
from oracle.oracle import OracleCase

pytestmark = pytest.mark.gpu

FORMS2 = {"fused": {"MPLBHIP_FUSED": "1"}, "tile": {"MPLBHIP_PAIR": "1"},
          "march": {"MPLBHIP_PAIR": "2"}}
FORMS3 = {"fused": {"MPLBHIP_FUSED": "1"}, "pair": {"MPLBHIP_PAIR": "1"}}
for k in range(4):
    FORMS3["fold%d" % k] = {"MPLBHIP_FUSED": "0", "MPLBHIP_XFACE_FOLD": str(k)}
    if k < 3:
        FORMS2["fold%d" % k] = FORMS3["fold%d" % k]
CASES = ([(2, f, s) for f in FORMS2 for s in (hip.STORE_F64, hip.STORE_F32, hip.STORE_F16)]
         + [(3, f, s) for f in FORMS3 for s in (hip.STORE_F64, hip.STORE_F32, hip.STORE_F16)]
         + [(3, "swap", hip.STORE_F64)])


@pytest.mark.parametrize("dim, form, storage", CASES)
def test_walls_read_incoming_populations_only(dim, form, storage, monkeypatch):
    print("%dD %s storage %d" % (dim, form, storage), flush=True)
    for k, v in (FORMS2 if dim == 2 else FORMS3).get(form, {}).items():
        monkeypatch.setenv(k, v)

    def build(be):
        if dim == 2:
            cases.cavity2d(be, 26)
        elif form == "swap":
            cases.cavity3d_swap(be, 20, size=(20, 13, 11))
        else:
            cases.cavity3d(be, 20, re=100.0, size=(20, 13, 11))

    o = OracleCase(dim)
    build(o)
    f = o.get_f(0)
    # one node of the left face and one of the face y = 0
    at = [(12, 0), (0, 9)] if dim == 2 else [(5, 6, 0), (4, 0, 9)]
    for i in at:
        f[(slice(None),) + i] = np.nan
    o.set_f(0, f)
    g = hip.LatticeCase(dim, storage=storage)
    build(g)
    g.set_f(0, f)
    for n in (1, 1, 2, 3):
        g.step(n)
        o.step(n)
        a, b = g.get_f(0), o.get_f(0)
        assert 0 < np.isnan(b).sum() < b.size
        if storage == hip.STORE_F64:
            assert np.array_equal(a, b, equal_nan=True), n
        else:
            assert np.array_equal(np.isnan(a), np.isnan(b)), n
    g.close()
