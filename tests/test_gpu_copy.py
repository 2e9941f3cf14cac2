"""Results handed to the host at the sizes where the copy changes: one staged
copy, the first size that goes through the ring, chunks that do not divide,
more chunks than slots (the ring is refilled), and a second copy on the same
context.  The same values through many small copies are the reference, bit
for bit: the copied quantity is the Gauss-point coordinates of a mesh, whose
subsets can be asked for one by one."""
import numpy as np
import pytest

from lowlevelfem import _lib
from lowlevelfem import mesh as M
from lowlevelfem import refelem as R

pytestmark = pytest.mark.gpu


# (cells, rule degree): 0.2 KB, 0.49 MB, 0.52 MB (above 512 KB), 4.7 MB, 24 MB, 187 MB of points
@pytest.mark.parametrize("cells,deg", [((1, 1, 1), 3), ((13, 14, 14), 3), ((13, 14, 15), 3), ((29, 29, 29), 3),
                                       ((32, 35, 33), 5), ((60, 60, 80), 5)])
def test_copy_sizes(gpu_ctx, cells, deg):
    m = M.structured_box_mesh(cells=cells)
    tab = R.rule_tables(m.etype, deg)
    dev = _lib.DeviceMesh(gpu_ctx, m.coords, m.etype, m.conn)
    for _ in range(2):
        P = dev.volume_points(tab)
        for sel in np.array_split(np.arange(m.E), max(1, m.E // 700))[::max(1, m.E // 30000)]:
            assert np.array_equal(P[sel], dev.volume_points(tab, sel))
    ref = np.einsum("qa,eai->eqi", tab.N, m.coords[m.conn[-50:]])
    assert np.abs(P[-50:] - ref).max() <= 1e-14
    dev.close()
