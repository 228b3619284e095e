"""ENO prolongation of fields that hold infinities, NaN, zeros of both signs,
denormals and values of the largest magnitude, whose products overflow: cell
kinds evaluate the two children between two cells together, and every choice of
a stencil and every fallback is the oracle's, per call and batched."""
import numpy as np
import pytest

import pyoracle as orc
from helpers import first_diff, host_array, same, sizes

cg = pytest.importorskip("carpet_amd")
pytestmark = pytest.mark.gpu

V, C = cg.VERTEX_CENTERED, cg.CELL_CENTERED
SPECIAL = np.array([np.inf, -np.inf, np.nan, 0.0, -0.0, 5e-324, -5e-324, 1e-160, 1.7e308, -1.7e308, 1e200])


def _dev(h):
    a = cg.DeviceArray(cg.Box(*h.box), padext=h.padext)
    a.upload(h.data)
    return a


@pytest.mark.parametrize("share", [0.002, 0.05, 0.5])
@pytest.mark.parametrize("cent,order,ntl", [(C, 5, 1), (C, 3, 1), (C, 5, 2), (C, 3, 3), (C, 5, 3), (V, 3, 1), (V, 3, 3)])
def test_special_values_match_oracle(cent, order, ntl, share):
    rng = np.random.default_rng(1000 + order + 10 * ntl + (cent == V))
    n = (75, 41, 33)
    s, lo, cs, co = (1, 5, 2, 0) if cent == V else (2, 11, 4, 2)
    reg = ((lo,) * 3, tuple(lo + (m - 1) * s for m in n), (s,) * 3)
    sb = ((co - 8 * cs,) * 3, tuple(co + (u // cs + 8) * cs for u in reg[1]), (cs,) * 3)
    db = (tuple(v - 2 * s for v in reg[0]), tuple(v + 3 * s for v in reg[1]), reg[2])
    srcs = []
    for _ in range(ntl):
        h = host_array(sb, sizes(sb))
        v = h.view()
        v[...] = rng.integers(-3, 4, size=v.shape)  # plateaus, ties and extrema beside the special values
        m = rng.random(v.shape) < share
        v[m] = rng.choice(SPECIAL, size=int(m.sum()))
        srcs.append(h)
    times = [0.0, -1.0, -2.0][:ntl]
    t = -0.5 if ntl > 1 else 0.0
    exp = host_array(db, sizes(db), 7.0)
    kind, o = (orc.KIND_VENO, 3) if cent == V else (orc.KIND_ENO, 3 if order == 5 else 2)
    assert orc.prolongate_time(kind, o, srcs, times, exp, t, reg, ntl - 1) == 0
    ds = [_dev(h) for h in srcs]
    for how in ("call", "batch"):
        d = _dev(host_array(db, sizes(db), 7.0))
        args = (d, ds, times, cg.Box(*reg), cg.Box(*reg), t, cg.OP_ENO, cent, order, ntl - 1)
        if how == "call":
            cg.transfer_from(*args)
        else:
            b = cg.Batch()
            b.add(0, *args)
            b.finalize()
            b.run()
        cg.synchronize()
        got = d.download_padded()
        assert same(got, exp.data), f"{how}: {first_diff(got, exp.data)}"
        if how == "batch":
            b.close()
