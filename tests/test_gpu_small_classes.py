"""Small prolongation regions of every tile shape run as one class on the 8x8
tiles, equal to the oracle bit for bit; a region too large for that keeps the
classes apart."""
import pytest

from helpers import first_diff, same
from workload_check import run_oracle

cg = pytest.importorskip("carpet_amd")
from carpet_amd.workloads import ArraySpec, Box, Transfer, Workload  # noqa: E402

pytestmark = pytest.mark.gpu

V, C = cg.VERTEX_CENTERED, cg.CELL_CENTERED


@pytest.mark.parametrize("large", [False, True])
@pytest.mark.parametrize("cent,op,order,ntl", [(V, cg.OP_LAGRANGE, 5, 3), (V, cg.OP_LAGRANGE, 3, 1),
                                               (C, cg.OP_LAGRANGE, 4, 2), (C, cg.OP_ENO, 5, 1), (V, cg.OP_ENO, 3, 3)])
def test_one_class_matches_oracle(cent, op, order, ntl, large):
    w = Workload("small classes")
    fs, cs, fo, co = (1, 2, 0, 0) if cent == V else (2, 4, 1, 2)
    cbox = Box((co - 6 * cs,) * 3, (co + 56 * cs,) * 3, (cs,) * 3)
    for tl in range(ntl):
        w.arrays[f"c{tl}"] = ArraySpec(cbox, seed=700 + tl)
    # thin in x, thin in x and y, a cube, one column wide, wide and flat
    ext = [(3, 50, 44), (6, 6, 40), (30, 30, 30), (1, 1, 1), (70, 20, 24), (64, 9, 31), (2, 60, 2)]
    ext = ext * 19  # 133 regions
    if large:
        ext.append((90, 80, 64))
    for r, n in enumerate(ext):
        lo = (5 + r % 19, 4 + r % 17, 3 + r % 2)
        reg = Box(tuple(fo + fs * l for l in lo), tuple(fo + fs * (l + k - 1) for l, k in zip(lo, n)), (fs,) * 3)
        w.arrays[f"f{r}"] = ArraySpec(reg.expand((3, 3, 3), (3, 3, 3)), owned=reg, seed=750 + r)
        w.steps.append(Transfer(f"f{r}", f"f{r}", [f"c{tl}" for tl in range(ntl)], [0.0, -1.0, -2.0][:ntl], reg, reg,
                                -0.5 if ntl > 1 else 0.0, op, cent, order, ntl - 1, phase=0))
        w.outputs.append(f"f{r}")
    ref = run_oracle(w)
    st = cg.Stream()
    dev = w.allocate()
    b = w.batch(dev)
    b.finalize()
    print(b.describe(), flush=True)
    if not large:
        assert b.launch_count() == 1 and "[tensor8 " in b.describe()
    else:
        assert b.launch_count() > 1
    b.run(st)
    st.synchronize()
    for k in ref:
        got = dev[k].download()
        if not same(got, ref[k]):
            raise AssertionError(f"{k} differs {first_diff(got, ref[k])}")
    b.close()
    w.free(dev)
