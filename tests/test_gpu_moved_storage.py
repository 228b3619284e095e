"""A batch's launch classes are those it was finalized with: new storage whose
rows start elsewhere in a 128-byte line changes which tile shape would suit a
region, and the tuner still times and rebuilds the same launches."""
import re

import numpy as np
import pytest

from helpers import first_diff, same
from workload_check import run_oracle

cg = pytest.importorskip("carpet_amd")
from carpet_amd.workloads import ArraySpec, Box, Transfer, Workload  # noqa: E402

pytestmark = pytest.mark.gpu


def _classes(b):
    return re.findall(r"^phase \d+ \[([^\]]+)\]", b.describe(), re.M)


@pytest.mark.parametrize("back", [False, True])
def test_autotune_after_the_alignment_changes(back, tmp_path):
    """160 x 32 points go to the 16x16-base tiles from a line's start and to the
    32x8 ones from its middle; 128 x 32 points always to the 32x8 ones."""
    w = Workload("moved")
    for tl in range(2):
        w.arrays[f"c{tl}"] = ArraySpec(Box((-16,) * 3, (200, 64, 64), (2,) * 3), seed=40 + tl)
    for nm, n in (("a", (160, 32, 24)), ("b", (128, 32, 24))):
        reg = Box((2, 2, 2), tuple(1 + k for k in n), (1,) * 3)
        w.arrays[nm] = ArraySpec(reg.expand((3,) * 3, (3,) * 3), owned=reg, seed=50 + n[0])
        w.steps.append(Transfer(nm, nm, ["c0", "c1"], [0.0, -1.0], reg, reg, -0.5, cg.OP_LAGRANGE,
                                cg.VERTEX_CENTERED, 3, 1, phase=0))
        w.outputs.append(nm)
    ref = run_oracle(w)
    st = cg.Stream()
    dev = w.allocate()
    moved, keep = {}, []
    for k in w.outputs:  # the regions' rows begin 3 + 5 points after a line
        a = dev[k]
        n = int(np.prod(a.padext))
        keep.append(cg.DeviceArray(Box((0, 0, 0), (n + 31, 0, 0), (1, 1, 1)), padext=(n + 32, 1, 1)))
        moved[k] = cg.DeviceArray.view(a.box, keep[-1].ptr + 8 * 5, a.padext)
    first, second = (moved, dev) if back else (dev, moved)
    b = w.batch({**dev, **first})
    b.finalize()
    classes = _classes(b)
    print(b.describe(), flush=True)
    assert len(classes) == (1 if back else 2)
    assert b.set_storage([(first[k], second[k]) for k in w.outputs]) == 2
    b.autotune(st, reps=1, cache_path=str(tmp_path / "tune.txt"))
    assert _classes(b) == classes
    for k in w.outputs:
        second[k].fill(np.nan, stream=st)
        second[k].fill_hash(w.arrays[k].seed, stream=st)
    b.run(st)
    st.synchronize()
    for k in ref:
        got = second[k].download()
        if not same(got, ref[k]):
            raise AssertionError(f"{k} differs {first_diff(got, ref[k])}")
    b.close()
    w.free(dev)
