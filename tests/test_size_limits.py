"""Regions whose planes have 2^32 points and more end in an error or in a
batch, never in a division by zero on the host: the plane's point count, cut to
32 bits, is the divisor of the kernels' index arithmetic."""
import subprocess
import sys
from pathlib import Path

import pytest

cg = pytest.importorskip("carpet_amd")

ROOT = Path(__file__).resolve().parent.parent

# one region of n points; the storage is never touched, the call is refused
CALL = """
import sys
sys.path.insert(0, {root!r})
from carpet_amd._lib import I3, lib
import carpet_amd as cg
n = {n}
e = I3(*n)
box = cg.Box((0, 0, 0), tuple(k - 1 for k in n), (1, 1, 1)).as_c()
at = 0x10000
rc = lib.cg_copy_3d_f64(at, e, e, at, e, e, box, box, box, box, None, None)
print("rc", rc, lib.cg_last_error_message().decode())
"""


@pytest.mark.parametrize("n", [(65536, 65536, 1), (131072, 65536, 2), (32768, 131072, 1), (65536, 32768, 1)])
def test_copy_of_a_huge_plane_is_refused(n):
    r = subprocess.run([sys.executable, "-c", CALL.format(root=str(ROOT), n=n)], capture_output=True, text=True,
                       timeout=120)
    assert r.returncode == 0, (r.returncode, r.stderr)
    assert "rc -1 region too large" in r.stdout, r.stdout


@pytest.mark.gpu
def test_tvd_batch_takes_a_huge_plane():
    """A TVD region of 65536 x 65536 x 2 fine points has 2^30 coarse parents,
    which fit a launch.  The batch is built and not run."""
    fine = cg.Box((1, 1, 1), (1 + 2 * 65535, 1 + 2 * 65535, 3), (2, 2, 2))
    coarse = cg.Box((2 - 4, 2 - 4, 2 - 4), (2 + 4 * 32768, 2 + 4 * 32768, 2 + 4), (4, 4, 4))
    own = cg.DeviceArray(cg.Box((0, 0, 0), (63, 0, 0), (1, 1, 1)))
    dst = cg.DeviceArray.view(fine, own.ptr, fine.sizes())
    src = cg.DeviceArray.view(coarse, own.ptr, coarse.sizes())
    b = cg.Batch()
    b.add(0, dst, [src], [0.0], fine, fine, 0.0, cg.OP_TVD, cg.CELL_CENTERED, 1, 0)
    b.finalize()
    assert f"items {2**30 // 1024} " in b.describe()
    b.close()


@pytest.mark.gpu
def test_copy_batch_refuses_a_huge_plane():
    box = cg.Box((0, 0, 0), (65535, 65535, 0), (1, 1, 1))
    own = cg.DeviceArray(cg.Box((0, 0, 0), (63, 0, 0), (1, 1, 1)))
    a = cg.DeviceArray.view(box, own.ptr, box.sizes())
    b = cg.Batch()
    b.add(0, a, [a], [0.0], box, box, 0.0, cg.OP_SYNC, cg.VERTEX_CENTERED, 1, 0)
    with pytest.raises(cg.CarpetError, match="too large"):
        b.finalize()
    b.close()
