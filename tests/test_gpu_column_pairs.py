"""FP32 arrays: classes whose regions' columns pair up run with two columns a
thread, all others with two rows.  Either way, and when new storage moves a
region of paired columns to an odd element, every point is the rounded FP64
oracle to one unit in the last place (the two FP64 results differ by
reassociation only), and nothing outside the region is written."""
import numpy as np
import pytest

import pyoracle as orc
from helpers import host_array, sizes

cg = pytest.importorskip("carpet_amd")
pytestmark = pytest.mark.gpu

V, C = cg.VERTEX_CENTERED, cg.CELL_CENTERED


def _ulps(a, b):
    def ordered(x):
        i = np.ascontiguousarray(x, dtype=np.float32).view(np.int32).astype(np.int64)
        return np.where(i < 0, -(i & 0x7FFFFFFF), i)
    return np.abs(ordered(a) - ordered(b))


def _case(cent, order, ntl, n, k):
    """Sources in [1, 2), the region, the destination box (k columns before the
    region) and the oracle's result on it, NaN outside the region."""
    s, lo, cs, co = (1, 4, 2, 0) if cent == V else (2, 9, 4, 2)
    reg = ((lo,) * 3, tuple(lo + (m - 1) * s for m in n), (s,) * 3)
    db = (tuple(l - s * (k if d == 0 else 1) for d, l in enumerate(reg[0])),
          tuple(u + s * (3 if d == 0 else 1) for d, u in enumerate(reg[1])), reg[2])
    sb = ((co - 8 * cs,) * 3, tuple(co + (u // cs + 8) * cs for u in reg[1]), (cs,) * 3)
    rng = np.random.default_rng(order * 100 + n[0])
    srcs = []
    for _ in range(ntl):
        h = host_array(sb, sizes(sb))
        h.view()[...] = (1 + rng.random(h.view().shape)).astype(np.float32)
        srcs.append(h)
    exp = host_array(db, sizes(db))
    kind = orc.KIND_VLAG if cent == V else orc.KIND_CLAG
    times = [1.0, 0.0, -1.0][:ntl]
    assert orc.prolongate_time(kind, order, srcs, times, exp, 1 / 3 if ntl > 1 else 1.0, reg, ntl - 1) == 0
    return srcs, times, cg.Box(*reg), cg.Box(*db), exp.view()


def _dev(h):
    a = cg.DeviceArray(cg.Box(*h.box), dtype=np.float32)
    a.upload(h.view().astype(np.float32))
    return a


def _padded(box, odd):
    e = box.sizes()
    pad = ((e[0] + 31) // 32 * 32 + odd, e[1], e[2])
    return pad, pad[0] * pad[1] * pad[2]


def _check(got, exp, what, dot2=False):
    """got: the padded destination, NaN before; exp: the oracle on the box"""
    full = np.full(got.shape, np.nan)
    full[:exp.shape[0], :exp.shape[1], :exp.shape[2]] = exp
    m = ~np.isnan(full)
    assert np.array_equal(m, ~np.isnan(got)), f"{what}: wrote outside the region, or not all of it"
    if dot2:
        assert cg.relative_errors(got[m].astype(np.float64), full[m])[0] <= 1e-6, what
    else:
        assert _ulps(got[m], full[m].astype(np.float32)).max() <= 1, what


@pytest.mark.parametrize("cent,order,ntl", [(V, 5, 3), (V, 3, 1), (C, 4, 2)])
@pytest.mark.parametrize("n,k,odd,columns", [(128, 0, 0, True), (126, 2, 0, True), (128, 0, 1, False), (127, 0, 0, False),
                                             (128, 1, 0, False), (125, 3, 0, False), (66, 0, 0, False), (1, 31, 0, False)])
def test_batch(cent, order, ntl, n, k, odd, columns):
    srcs, times, reg, box, exp = _case(cent, order, ntl, (n, 20, 12), k)
    ds = [_dev(h) for h in srcs]
    pad, count = _padded(box, odd)
    own = cg.DeviceArray(cg.Box((0, 0, 0), (count + 63, 0, 0), (1, 1, 1)), dtype=np.float32, padext=(count + 64, 1, 1))
    for prec in (cg.PREC_MIXED, cg.PREC_MIXED_DOT2):
        b = cg.Batch()
        at = {s: cg.DeviceArray.view(box, own.ptr + 4 * s, pad, np.float32) for s in (0, 1, 33)}
        b.add(0, at[0], ds, times, reg, reg, 1 / 3 if ntl > 1 else 1.0, cg.OP_LAGRANGE, cent, order, ntl - 1, prec=prec)
        b.finalize()
        assert (" columns" in b.describe()) == (columns and prec == cg.PREC_MIXED), b.describe()
        last = 0
        for s in (0, 1, 33):
            if s != last:
                assert b.set_storage([(at[last], at[s])]) == 1
            last = s
            own.upload(np.full((1, 1, count + 64), np.nan, np.float32))
            b.run()
            cg.synchronize()
            flat = own.download().ravel()
            assert np.isnan(flat[:s]).all() and np.isnan(flat[s + count:]).all()
            _check(flat[s:s + count].reshape(pad[::-1]), exp, f"prec {prec} at {s}", prec == cg.PREC_MIXED_DOT2)
        b.close()


@pytest.mark.parametrize("n,k", [(256, 0), (256, 1), (257, 2)])
def test_call(n, k):
    srcs, times, reg, box, exp = _case(V, 3, 1, (n, 256, 256), k)
    ds = [_dev(h) for h in srcs]
    pad, _ = _padded(box, 0)
    dd = cg.DeviceArray(box, dtype=np.float32, padext=pad)
    dd.upload(np.full(exp.shape, np.nan, np.float32), fill=np.nan)
    cg.transfer_from_mixed(dd, ds, times, reg, reg, 1.0, cg.OP_LAGRANGE, V, 3, 0)
    cg.synchronize()
    _check(dd.download_padded(), exp, "call")


@pytest.mark.parametrize("cent,order,ntl,n,k,columns", [(V, 7, 1, 66, 0, True), (C, 5, 2, 66, 2, True), (V, 5, 3, 66, 1, False),
                                                        (V, 9, 1, 65, 0, False), (C, 4, 1, 66, 0, False)])
def test_narrow_tiles_of_large_classes(cent, order, ntl, n, k, columns):
    srcs, times, reg, box, exp = _case(cent, order, ntl, (n, 101, 161), k)
    ds = [_dev(h) for h in srcs]
    pad, count = _padded(box, 0)
    own = cg.DeviceArray(cg.Box((0, 0, 0), (count + 31, 0, 0), (1, 1, 1)), dtype=np.float32, padext=(count + 32, 1, 1))
    at = {s: cg.DeviceArray.view(box, own.ptr + 4 * s, pad, np.float32) for s in (0, 1)}
    b = cg.Batch()
    b.add(0, at[0], ds, times, reg, reg, 1 / 3 if ntl > 1 else 1.0, cg.OP_LAGRANGE, cent, order, ntl - 1, prec=cg.PREC_MIXED)
    b.finalize()
    d = b.describe()
    assert "tensorN" in d and (" columns" in d) == columns, d
    for s in (0, 1):
        if s:
            assert b.set_storage([(at[0], at[1])]) == 1
        own.upload(np.full((1, 1, count + 32), np.nan, np.float32))
        b.run()
        cg.synchronize()
        flat = own.download().ravel()
        assert np.isnan(flat[:s]).all() and np.isnan(flat[s + count:]).all()
        _check(flat[s:s + count].reshape(pad[::-1]), exp, f"at {s}")
    b.close()
