"""Single prolongations of the sizes at which their z chunks change -- short
chunks of few tiles, chunks kept long where shorter ones would share the CUs,
chunks stretched to fit one round of workgroups -- equal the oracle."""
import pytest

from helpers import first_diff, same
from workload_check import run_oracle

cg = pytest.importorskip("carpet_amd")
from carpet_amd.workloads import ArraySpec, Box, Transfer, Workload  # noqa: E402

pytestmark = pytest.mark.gpu

V, C = cg.VERTEX_CENTERED, cg.CELL_CENTERED


@pytest.mark.parametrize("cent,op,order,ntl,n", [
    (V, cg.OP_LAGRANGE, 3, 1, (30, 20, 9)), (V, cg.OP_LAGRANGE, 5, 3, (66, 66, 67)),
    (V, cg.OP_LAGRANGE, 7, 1, (220, 220, 221)), (V, cg.OP_LAGRANGE, 11, 3, (150, 150, 75)),
    (V, cg.OP_LAGRANGE, 5, 3, (300, 316, 157)), (C, cg.OP_LAGRANGE, 5, 3, (220, 110, 219)),
    (C, cg.OP_ENO, 5, 3, (256, 200, 60)), (V, cg.OP_ENO, 3, 1, (180, 179, 181))])
def test_chunks_match_oracle(cent, op, order, ntl, n):
    w = Workload("chunks")
    fs, cs, fo, co = (1, 2, 0, 0) if cent == V else (2, 4, 1, 2)
    cbox = Box((co - 6 * cs,) * 3, tuple(co + (k // 2 + 12) * cs for k in n), (cs,) * 3)
    for tl in range(ntl):
        w.arrays[f"c{tl}"] = ArraySpec(cbox, seed=400 + tl)
    lo = (5, 4, 3)
    reg = Box(tuple(fo + fs * l for l in lo), tuple(fo + fs * (l + k - 1) for l, k in zip(lo, n)), (fs,) * 3)
    w.arrays["f"] = ArraySpec(reg.expand((3,) * 3, (3,) * 3), owned=reg, seed=450)
    w.steps.append(Transfer("f", "f", [f"c{tl}" for tl in range(ntl)], [0.0, -1.0, -2.0][:ntl], reg, reg,
                            -0.5 if ntl > 1 else 0.0, op, cent, order, ntl - 1, phase=0))
    w.outputs.append("f")
    ref = run_oracle(w)
    st = cg.Stream()
    dev = w.allocate()
    w.run_steps(dev, st)
    st.synchronize()
    got = dev["f"].download()
    if not same(got, ref["f"]):
        raise AssertionError(f"f differs {first_diff(got, ref['f'])}")
    w.free(dev)
