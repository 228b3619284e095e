"""How a batch cuts its transfers into work items: rows of operators that compute
much per point have no idle slots, the segments of the eight XCDs hold equal
numbers of items, classes that fit one round of workgroups take one each, and
the tiles of a row are no more than they have to be."""
import re

import pytest

cg = pytest.importorskip("carpet_amd")
from carpet_amd.workloads import Box  # noqa: E402

pytestmark = pytest.mark.gpu

V, C = cg.VERTEX_CENTERED, cg.CELL_CENTERED


def _launches(b):
    """items, grid, zchunk, points per item and mode of every launch"""
    return [tuple(map(int, m)) for m in
            re.findall(r"\] items (\d+) grid (\d+) zchunk (\d+) pt (\d+) wpc (-?\d+)", b.describe())]


def _array(box, first=0, pad=16):
    """A view whose element (0,0,0) lies `first` elements after a 128-byte line
    and whose rows are padded to a multiple of `pad`.  Its storage is not large
    enough: the batches here are built, not run."""
    e = box.sizes()
    return cg.DeviceArray.view(box, _base().ptr + 8 * first, ((e[0] + pad - 1) // pad * pad, e[1], e[2]))


_own = []


def _base():
    if not _own:
        _own.append(cg.DeviceArray(Box((0, 0, 0), (255, 0, 0), (1, 1, 1))))
    return _own[0]


def _prolong(b, n, cent, op, order, ntl=1, first=0, pad=16):
    s, lo, h = (1, 2, 8) if cent == V else (2, 1, 8)
    reg = Box((lo,) * 3, tuple(lo + (k - 1) * s for k in n), (s,) * 3)
    up = tuple(u // (2 * s) for u in reg.upper)
    src = Box((-2 * h,) * 3, tuple(2 * (u + h) for u in up), (2,) * 3) if cent == V else \
        Box((2 - 4 * h,) * 3, tuple(2 + 4 * (u + h) for u in up), (4,) * 3)
    d, a = _array(reg, first, pad), _array(src)
    b.add(0, d, [a] * ntl, [0.0, -1.0, -2.0][:ntl], reg, reg, -0.5 if ntl > 1 else 0.0, op, cent, order, ntl - 1)


def _restrict(b, n, first, op=cg.OP_LAGRANGE, cent=C):
    if cent == C:
        src = Box((1,) * 3, tuple(1 + 2 * (2 * k + 24) for k in n), (2,) * 3)
        reg = Box((18,) * 3, tuple(18 + 4 * (k - 1) for k in n), (4,) * 3)
    else:
        src = Box((0,) * 3, tuple(2 * k + 24 for k in n), (1,) * 3)
        reg = Box((8,) * 3, tuple(8 + 2 * (k - 1) for k in n), (2,) * 3)
    b.add(0, _array(reg, first), [_array(src)], [0.0], reg, reg, 0.0, op, cent, 1, 0)


@pytest.mark.parametrize("what,idle", [("stagger3", False), ("stagger2", False), ("restrict_stagger", False),
                                       ("cc_o3", False), ("cc_o5", False), ("monotone", False), ("average", True)])
def test_rows_of_costly_operators_have_no_idle_slots(what, idle):
    """Rows of 17 points that begin 8 points into a line."""
    n = (17, 40, 40)
    cg.set_staggered_operators(True)
    cg.set_restriction(what in ("cc_o3", "cc_o5"), 5 if what == "cc_o5" else 3)
    try:
        b = cg.Batch()
        if what.startswith("stagger"):
            _prolong(b, n, V, cg.OP_STAGGER111, int(what[-1]), first=8)
        elif what == "monotone":
            _prolong(b, n, V, cg.OP_LAGRANGE_MONOTONE, 5, first=8)
        else:
            st = what == "restrict_stagger"
            _restrict(b, n, 8, cg.OP_STAGGER111 if st else cg.OP_LAGRANGE, V if st else C)
        b.finalize()
    finally:
        cg.set_staggered_operators(False)
        cg.set_restriction(False, 3)
    items, _, _, pt, _ = _launches(b)[0]
    slots = (32 if idle else 17) * 40 * 40
    assert items == (slots + pt - 1) // pt, b.describe()
    b.close()


@pytest.mark.parametrize("n,count", [((112, 112, 112), 24), ((260, 256, 256), 8)])
def test_tvd_items_are_even_over_the_xcds(n, count):
    """Many medium regions, which are cut into slabs, and a gigabyte of large ones,
    which go to the XCDs in blocks of 64 items: the longest of the eight
    segments, an eighth of the grid, holds at most 64 items more than the mean."""
    b = cg.Batch()
    for _ in range(count):
        _prolong(b, n, C, cg.OP_TVD, 1)
    b.finalize()
    items, grid, _, _, wpc = _launches(b)[0]
    assert items == count * -(-n[0] * n[1] * n[2] // 8192)
    assert wpc == -1
    assert grid / 8 <= items / 8 + 64, b.describe()
    b.close()


@pytest.mark.parametrize("n,count,ntl,order", [((250, 120, 120), 4, 3, 11), ((250, 120, 120), 4, 3, 9)])
def test_a_class_of_one_round_spreads_evenly(n, count, ntl, order):
    """Items of about equal cost that just fit the resident workgroups: no XCD's
    segment is longer than it holds at once."""
    b = cg.Batch()
    for _ in range(count):
        _prolong(b, n, V, cg.OP_LAGRANGE, order, ntl, first=8)
    b.finalize()
    d = b.describe()
    items, grid, _, _, wpc = _launches(b)[0]
    assert wpc == 0 and "one round" in d, d
    assert items <= grid < items + 8 * count, d
    b.close()


def test_a_class_of_one_round_with_three_workgroups_to_a_cu_keeps_equal_cost():
    """Regions whose last z chunk is short: the segments of equal cost differ by
    more items than there are regions."""
    b = cg.Batch()
    for _ in range(6):
        _prolong(b, (67, 145, 161), V, cg.OP_ENO, 3, 2, first=8)
    b.finalize()
    d = b.describe()
    items, grid, _, _, wpc = _launches(b)[0]
    assert wpc == 0 and "one round" in d, d
    assert grid >= items + 8 * 6, d
    b.close()


@pytest.mark.parametrize("cent,op,order,ntl,n,first,pad,tiles", [
    (V, cg.OP_LAGRANGE, 5, 1, 250, 8, 16, 5),  # cheap: the line, for a quarter more tiles
    (V, cg.OP_LAGRANGE, 5, 3, 250, 8, 16, 4),  # the half line
    (V, cg.OP_LAGRANGE, 5, 3, 256, 4, 16, 5),  # unaligned but for one more tile
    (C, cg.OP_ENO, 5, 3, 256, 4, 16, 4),  # expensive: no more tiles
    (V, cg.OP_ENO, 3, 3, 256, 12, 16, 4),
    (V, cg.OP_LAGRANGE, 5, 1, 250, 8, 1, 4),  # rows that lose their place in a line
    (V, cg.OP_LAGRANGE, 3, 1, 250, 8, 2, 4),
    (V, cg.OP_LAGRANGE, 5, 1, 248, 12, 8, 4),  # rows that keep their place in a half line
])
def test_tiles_along_x(cent, op, order, ntl, n, first, pad, tiles):
    b = cg.Batch()
    _prolong(b, (n, 112, 120), cent, op, order, ntl, first=first, pad=pad)
    b.finalize(60)
    d = b.describe()
    assert "[tensor " in d, d
    items = _launches(b)[0][0]
    assert items in [tiles * rows * chunks for rows in (7, 8) for chunks in (1, 2)], d
    b.close()
