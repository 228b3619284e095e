"""Tensor tiles and the rows of pointwise operators start at a 128-byte line of
the destination: regions at every offset from a line, of widths around the
tiles' and lines' and of both parities, per call and batched, equal the oracle
bit for bit."""
import numpy as np
import pytest

from helpers import first_diff, same
from workload_check import run_oracle

cg = pytest.importorskip("carpet_amd")
from carpet_amd.workloads import ArraySpec, Box, Transfer, Workload, hash_field  # noqa: E402

pytestmark = pytest.mark.gpu

V, C = cg.VERTEX_CENTERED, cg.CELL_CENTERED


def _regions(cent, op, order, ntl, ny, nz):
    """One destination array per region: its first column lies k points after
    the owned interior's, which the padding puts on a line."""
    w = Workload("aligned")
    s = 1 if cent == V else 2
    times = [0.0, -1.0, -2.0][:ntl]
    for tl in range(ntl):
        if cent == V:
            cbox = Box((-16,) * 3, (200, 64, 64), (2,) * 3)
        else:
            cbox = Box((2 - 32,) * 3, (402, 130, 130), (4,) * 3)
        w.arrays[f"c{tl}"] = ArraySpec(cbox, seed=40 + tl)
    lo = 2 if cent == V else 1
    for i, n in enumerate((1, 2, 5, 15, 16, 17, 31, 33, 63, 64, 65, 80, 130)):
        for k in ((i * 7) % 16, (i * 5 + 1) % 16, 17):
            own = Box((lo, lo, lo), (lo + 150 * s, lo + 45 * s, lo + 30 * s), (s,) * 3)
            reg = Box((lo + k * s, lo + s, lo), (lo + (k + n - 1) * s, lo + ny * s, lo + (nz - 1) * s), (s,) * 3)
            nm = f"d{n}_{k}"
            w.arrays[nm] = ArraySpec(own.expand((2, 1, 1), (2, 1, 1)), owned=own, seed=900 + 31 * n + k)
            w.steps.append(Transfer(nm, nm, [f"c{tl}" for tl in range(ntl)], times, reg, reg, -0.5 if ntl > 1 else 0.0,
                                    op, cent, order, ntl - 1, phase=0))
            w.outputs.append(nm)
    return w


@pytest.mark.parametrize("ny,nz", [(40, 20), (5, 4), (37, 3)])
@pytest.mark.parametrize("cent,op,order,ntl", [(V, cg.OP_LAGRANGE, 1, 1), (V, cg.OP_LAGRANGE, 3, 2),
                                               (V, cg.OP_LAGRANGE, 5, 3), (V, cg.OP_LAGRANGE, 11, 1),
                                               (C, cg.OP_LAGRANGE, 0, 1), (C, cg.OP_LAGRANGE, 2, 2),
                                               (C, cg.OP_LAGRANGE, 4, 1), (C, cg.OP_LAGRANGE, 5, 3),
                                               (C, cg.OP_ENO, 3, 1), (C, cg.OP_ENO, 5, 3), (V, cg.OP_ENO, 3, 3)])
def test_offsets_match_oracle(cent, op, order, ntl, ny, nz):
    w = _regions(cent, op, order, ntl, ny, nz)
    ref = run_oracle(w)
    st = cg.Stream()
    for how in ("per call", "batched"):
        dev = w.allocate()
        if how == "per call":
            w.run_steps(dev, st)
        else:
            b = w.batch(dev)
            b.finalize()
            b.run(st)
        st.synchronize()
        for k in ref:
            got = dev[k].download()
            if not same(got, ref[k]):
                raise AssertionError(f"{how}: {k} differs {first_diff(got, ref[k])}")
        if how == "batched":
            b.close()
        w.free(dev)


def _point_regions(what, ny, nz):
    """As _regions, for copies, injections and cell restrictions, and a same-
    level time interpolation."""
    w = Workload(what)
    s, cent = {"copy": (1, V), "interp": (1, V), "inject": (2, V), "average": (4, C)}[what]
    lo = 4 if cent == V else 2
    srcs = ["a", "b"] if what == "interp" else ["a"]
    f = s if what in ("copy", "interp") else s // 2
    for i, nm in enumerate(srcs):
        if what in ("copy", "interp"):
            sbox = Box((lo - 3,) * 3, (lo + 190, lo + 60, lo + 40), (1,) * 3)
        elif cent == V:
            sbox = Box((0,) * 3, (360, 110, 70), (f,) * 3)
        else:
            sbox = Box((1,) * 3, (1 + 2 * 360, 1 + 2 * 110, 1 + 2 * 70), (f,) * 3)
        w.arrays[nm] = ArraySpec(sbox, seed=60 + i)
    for i, n in enumerate((1, 3, 7, 8, 15, 16, 17, 31, 33, 64, 65, 100, 130)):
        for k in ((i * 7) % 16, (i * 5 + 1) % 16, 17):
            own = Box((lo, lo, lo), (lo + 150 * s, lo + 45 * s, lo + 30 * s), (s,) * 3)
            reg = Box((lo + k * s, lo + s, lo), (lo + (k + n - 1) * s, lo + ny * s, lo + (nz - 1) * s), (s,) * 3)
            nm = f"d{n}_{k}"
            w.arrays[nm] = ArraySpec(own.expand((2, 1, 1), (2, 1, 1)), owned=own, seed=300 + 31 * n + k)
            t = ([0.0, -1.0], -0.25) if what == "interp" else ([0.0], 0.0)
            w.steps.append(Transfer(nm, nm, srcs, t[0], reg, reg, t[1], cg.OP_LAGRANGE, cent, 1, len(srcs) - 1, phase=0))
            w.outputs.append(nm)
    return w


@pytest.mark.parametrize("ny,nz", [(40, 20), (3, 3), (1, 1)])
@pytest.mark.parametrize("what", ["copy", "interp", "inject", "average"])
def test_point_offsets_match_oracle(what, ny, nz):
    w = _point_regions(what, ny, nz)
    ref = run_oracle(w)
    st = cg.Stream()
    for how in ("per call", "batched", "moved"):
        dev = w.allocate()
        keep = []
        if how == "per call":
            w.run_steps(dev, st)
        else:
            b = w.batch(dev)
            b.finalize()
            if how == "moved":  # storage whose rows start elsewhere in a line
                for k in w.outputs:
                    a = dev[k]
                    n = int(np.prod(a.padext))
                    keep.append((a, cg.DeviceArray(Box((0, 0, 0), (n + 31, 0, 0), (1, 1, 1)), padext=(n + 32, 1, 1))))
                    m = cg.DeviceArray.view(a.box, keep[-1][1].ptr + 8 * 5, a.padext)
                    m.fill(np.nan, stream=st)
                    m.fill_hash(w.arrays[k].seed, stream=st)
                    b.set_storage([(a, m)])
                    dev[k] = m
            b.run(st)
        st.synchronize()
        for k in ref:
            got = dev[k].download()
            if not same(got, ref[k]):
                raise AssertionError(f"{how}: {k} differs {first_diff(got, ref[k])}")
        if how != "per call":
            b.close()
        w.free(dev)


@pytest.mark.parametrize("prec", [cg.PREC_MIXED, cg.PREC_MIXED_DOT2])
def test_float_storage_does_not_depend_on_the_offset(prec):
    """FP32 rows hold 32 points a line: the same region gives the same values
    wherever its rows start."""
    cbox = Box((-16,) * 3, (200, 64, 64), (2,) * 3)
    reg = Box((3, 2, 2), (152, 31, 20), (1,) * 3)
    src = []
    for tl in range(3):
        a = cg.DeviceArray(cbox, dtype=np.float32)
        a.upload(hash_field(70 + tl, cbox.sizes()))
        src.append(a)
    outs = []
    for k in (0, 1, 2, 15, 16, 17, 31):
        box = reg.expand((k, 0, 0), (3, 0, 0))
        d = cg.DeviceArray(box, dtype=np.float32, padext=(box.sizes()[0] + 1,) + box.sizes()[1:])
        d.upload(np.zeros((box.sizes()[2], box.sizes()[1], box.sizes()[0]), np.float32))
        b = cg.Batch()
        b.add(0, d, src, [0.0, -1.0, -2.0], reg, reg, -0.5, cg.OP_LAGRANGE, V, 5, 2, prec=prec)
        b.finalize()
        b.run()
        cg.synchronize()
        outs.append(d.download()[:, :, k:k + reg.sizes()[0]])
        b.close()
    for o in outs[1:]:
        assert same(o, outs[0]), first_diff(o, outs[0])


def test_storage_of_another_alignment():
    """New storage keeps the items a class was finalized with, also where its
    rows start elsewhere in a line."""
    w = _regions(V, cg.OP_LAGRANGE, 5, 3, 40, 20)
    ref = run_oracle(w)
    st = cg.Stream()
    dev = w.allocate()
    b = w.batch(dev)
    b.finalize()
    for shift in (1, 9):
        moved, keep = {}, []
        for k in w.outputs:
            a = dev[k]
            n = int(np.prod(a.padext))
            own = cg.DeviceArray(Box((0, 0, 0), (n + 31, 0, 0), (1, 1, 1)), padext=(n + 32, 1, 1))
            keep.append(own)
            m = cg.DeviceArray.view(a.box, own.ptr + 8 * shift, a.padext)
            m.fill(np.nan, stream=st)
            m.fill_hash(w.arrays[k].seed, stream=st)
            moved[k] = m
        assert b.set_storage([(dev[k], moved[k]) for k in w.outputs]) == len(w.steps)
        b.run(st)
        st.synchronize()
        for k in ref:
            got = moved[k].download()
            if not same(got, ref[k]):
                raise AssertionError(f"shift {shift}: {k} differs {first_diff(got, ref[k])}")
        assert b.set_storage([(moved[k], dev[k]) for k in w.outputs]) == len(w.steps)
    b.close()
    w.free(dev)
