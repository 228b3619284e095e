"""A phase of many small regions runs as one launch, unless the caller named how
its launches run before the batch was finalized: then its classes stay apart,
side by side or in turn as asked, with the same results."""
import pytest

from helpers import first_diff, same
from workload_check import run_oracle

cg = pytest.importorskip("carpet_amd")
from carpet_amd.workloads import ArraySpec, Box, Transfer, Workload  # noqa: E402

pytestmark = pytest.mark.gpu


def test_a_named_mode_keeps_the_classes():
    w = Workload("named modes")
    for tl in range(2):
        w.arrays[f"c{tl}"] = ArraySpec(Box((-12,) * 3, (112,) * 3, (2,) * 3), seed=700 + tl)
    ext = [(3, 50, 44), (6, 6, 40), (30, 30, 30), (1, 1, 1), (70, 20, 24), (64, 9, 31), (2, 60, 2)] * 19
    for r, n in enumerate(ext * 2):  # two phases of 133 regions
        lo = (5 + r % 19, 4 + r % 17, 3 + r % 2)
        reg = Box(lo, tuple(l + k - 1 for l, k in zip(lo, n)), (1,) * 3)
        w.arrays[f"f{r}"] = ArraySpec(reg.expand((3, 3, 3), (3, 3, 3)), owned=reg, seed=750 + r)
        w.steps.append(Transfer(f"f{r}", f"f{r}", ["c0", "c1"], [0.0, -1.0], reg, reg, -0.5, cg.OP_LAGRANGE,
                                cg.VERTEX_CENTERED, 3, 1, phase=r // len(ext)))
        w.outputs.append(f"f{r}")
    ref = run_oracle(w)
    st = cg.Stream()
    for mode, words in ((1, "side by side"), (0, "in turn")):
        dev = w.allocate()
        b = w.batch(dev)
        b.set_phase_mode(1, mode)
        b.finalize()
        lines = [x for x in b.describe().splitlines() if x.startswith("phase ")]
        first, second = ([x for x in lines if x.startswith(f"phase {p} ")] for p in (0, 1))
        assert len(first) == 1 and len(second) > 1, lines
        assert all(x.endswith(words) for x in second), lines
        b.run(st)
        st.synchronize()
        for k in ref:
            got = dev[k].download()
            if not same(got, ref[k]):
                raise AssertionError(f"mode {mode}: {k} differs {first_diff(got, ref[k])}")
        b.close()
        w.free(dev)
