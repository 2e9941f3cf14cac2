"""Body force over part of the elements, with components that are not finite:
a node that no element of the set touches gets exactly 0, as the sum over no
element; the finite component is not touched by the others."""
import numpy as np
import pytest

from lowlevelfem import _lib
from lowlevelfem import mesh as M
from lowlevelfem import refelem as R

pytestmark = pytest.mark.gpu


# a thread per element (8 and 10 nodes) and a wavefront per element (27)
@pytest.mark.parametrize("elem,order,cells", [("hex", 1, (4, 3, 5)), ("tet", 2, (2, 3, 2)), ("hex", 2, (2, 2, 3))])
@pytest.mark.parametrize("count", [0, 1, 0.5])
def test_force_outside_the_set(gpu_ctx, elem, order, cells, count):
    m = M.structured_box_mesh(cells=cells, elem=elem, order=order)
    tab = R.rule_tables(m.etype, 2 * order + 1)
    dev = _lib.DeviceMesh(gpu_ctx, m.coords, m.etype, m.conn)
    sel = np.arange(count if isinstance(count, int) else m.E // 2)
    touched = np.zeros(m.N, bool)
    touched[np.asarray(m.conn)[sel].ravel()] = True
    f = dev.body(tab, g=[np.inf, np.nan, 1.5], elems=sel).reshape(-1, 3)
    assert not f[~touched].any()
    assert not np.isfinite(f[touched][:, :2]).any()
    assert np.array_equal(f[:, 2], dev.body(tab, g=[0.0, 0.0, 1.5], elems=sel).reshape(-1, 3)[:, 2])
    dev.close()
