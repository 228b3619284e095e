"""The launch modes of tensor classes over several rounds of workgroups: counters
(wpc 0 and 2), fixed rounds (wpc -2), and one workgroup per item (wpc -1), each
equal to the oracle; a phase with a class that takes its items from counters by
default runs its launches in turn."""
import re

import numpy as np
import pytest

from helpers import first_diff, same
from workload_check import run_oracle

cg = pytest.importorskip("carpet_amd")
from carpet_amd.workloads import ArraySpec, Box, Transfer, Workload  # noqa: E402

pytestmark = pytest.mark.gpu

V, C = cg.VERTEX_CENTERED, cg.CELL_CENTERED
HOW = {-1: "one per item", 0: "counters", 2: "counters", -2: "fixed rounds"}


def _workload(cent, op, order, ntl, exts):
    """Prolongations from one coarse array onto regions of the given extents."""
    w = Workload("modes")
    fs, cs, fo, co = (1, 2, 0, 0) if cent == V else (2, 4, 1, 2)
    top = max(max(e) for e in exts) // 2 + 24
    for tl in range(ntl):
        w.arrays[f"c{tl}"] = ArraySpec(Box((co - 6 * cs,) * 3, (co + top * cs,) * 3, (cs,) * 3), seed=800 + tl)
    for r, n in enumerate(exts):
        lo = (5 + r % 19, 4 + r % 17, 3 + r % 2)
        reg = Box(tuple(fo + fs * l for l in lo), tuple(fo + fs * (l + k - 1) for l, k in zip(lo, n)), (fs,) * 3)
        w.arrays[f"f{r}"] = ArraySpec(reg.expand((3,) * 3, (3,) * 3), owned=reg, seed=850 + r)
        w.steps.append(Transfer(f"f{r}", f"f{r}", [f"c{tl}" for tl in range(ntl)], [0.0, -1.0, -2.0][:ntl], reg, reg,
                                -0.5 if ntl > 1 else 0.0, op, cent, order, ntl - 1, phase=0))
        w.outputs.append(f"f{r}")
    return w


def _check(w, dev, ref, what):
    for k in ref:
        got = dev[k].download()
        if not same(got, ref[k]):
            raise AssertionError(f"{what}: {k} differs {first_diff(got, ref[k])}")


def _poison(w, dev, st):
    for k in w.outputs:
        dev[k].fill(np.nan, stream=st)
        dev[k].fill_hash(w.arrays[k].seed, stream=st)


@pytest.mark.parametrize("cent,op,order,ntl", [(V, cg.OP_LAGRANGE, 5, 3), (C, cg.OP_LAGRANGE, 4, 2),
                                               (C, cg.OP_ENO, 5, 3), (V, cg.OP_ENO, 3, 2)])
def test_modes_over_several_rounds(cent, op, order, ntl, tmp_path):
    w = _workload(cent, op, order, ntl, [(60, 50, 40)] * 64)
    ref = run_oracle(w)
    st = cg.Stream()
    dev = w.allocate()
    b = w.batch(dev)
    b.finalize()
    keys = re.findall(r"\[([^\]]+)\]", b.describe())
    assert len(keys) == 1
    for wpc, how in HOW.items():
        cache = tmp_path / f"t{wpc}.txt"
        cache.write_text(f"{keys[0]}|2 4096 {wpc} -1 1\n")
        b.autotune(st, reps=1, cache_path=str(cache))
        d = b.describe()
        items, grid = map(int, re.search(r"items (\d+) grid (\d+)", d).groups())
        print(d, flush=True)
        assert f"wpc {wpc} " in d and how in d
        assert items > 2 * grid if wpc != -1 else grid >= items
        _poison(w, dev, st)
        b.run(st)
        st.synchronize()
        _check(w, dev, ref, f"wpc {wpc}")
    b.close()
    w.free(dev)


def test_phase_with_a_counter_class_runs_in_turn():
    """A region of more than 2^25 points in tiles of 4 planes takes its items
    from counters; thin faces beside it, one workgroup per item."""
    w = _workload(V, cg.OP_LAGRANGE, 1, 1, [(324, 324, 324), (3, 80, 66), (6, 56, 42)])
    ref = run_oracle(w)
    st = cg.Stream()
    dev = w.allocate()
    b = w.batch(dev)
    b.finalize(4)
    d = b.describe()
    print(d, flush=True)
    assert re.search(r"\[tensor k0 o1 t1 [^\]]*\] .* wpc 0 .* counters in turn", d), d
    assert re.search(r"\[tensor4 [^\]]*\] .* wpc -1 .* one per item in turn", d), d
    items, grid = map(int, re.search(r"\[tensor k0 [^\]]*\] items (\d+) grid (\d+)", d).groups())
    assert items > 2 * grid
    b.run(st)
    st.synchronize()
    _check(w, dev, ref, "in turn")
    b.set_phase_mode(0, 1)
    assert "side by side" in b.describe()
    _poison(w, dev, st)
    b.run(st)
    st.synchronize()
    _check(w, dev, ref, "side by side")
    b.close()
    w.free(dev)
