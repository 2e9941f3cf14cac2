"""Body-force kernels at the sizes where they change: one thread per element
(4, 6, 8, 10 nodes; fewer and more elements than a block), one wavefront per
element (27 and 125 nodes), rules of up to and above the 64 points a
wavefront takes at once, element subsets and the empty set, against the CPU
oracle.  FP64 sums of some hundred terms of one sign and size per node: 1e-13
of the largest entry."""
import numpy as np
import pytest

from lowlevelfem import _lib
from lowlevelfem import mesh as M
from lowlevelfem import refelem as R
from oracle import oracle as O

pytestmark = pytest.mark.gpu

CASES = [("tet", 1, (1, 1, 1), 3), ("tet", 1, (4, 4, 3), 3), ("prism", 1, (3, 3, 3), 3), ("hex", 1, (9, 8, 4), 3),
         ("hex", 1, (2, 2, 2), 9), ("tet", 2, (4, 3, 4), 5), ("hex", 2, (3, 2, 2), 5), ("hex", 2, (2, 1, 3), 7),
         ("hex", 2, (1, 2, 1), 9), ("hex", 4, (1, 1, 2), 9)]


@pytest.mark.parametrize("elem,order,cells,deg", CASES)
def test_body(gpu_ctx, elem, order, cells, deg):
    m = M.structured_box_mesh(cells=cells, elem=elem, order=order, perturb=0.05, seed=3)
    tab = R.rule_tables(m.etype, deg)
    dev = _lib.DeviceMesh(gpu_ctx, m.coords, m.etype, m.conn)
    g = np.array([0.7, -1.1, 0.3])

    def close(a, b):
        return np.abs(a - b).max() <= 1e-13 * np.abs(b).max()

    assert close(dev.body(tab, g=g), O.body_force(m, tab, g))
    rng = np.random.default_rng(4)
    sel = rng.permutation(m.E)[:max(1, m.E // 2)]
    assert close(dev.body(tab, g=g, elems=sel), O.body_force(m, tab, g, elems=sel))
    G = rng.uniform(0.5, 1.5, (m.E, tab.q, 3))
    assert close(dev.body(tab, g_gp=G), O.body_force(m, tab, g_gp=G))
    assert close(dev.body(tab, g_gp=G[:sel.size], elems=sel), O.body_force(m, tab, g_gp=G[:sel.size], elems=sel))
    none = np.zeros(0, dtype=np.int64)
    assert not dev.body(tab, g=g, elems=none).any()
    assert np.allclose(dev.volume_points(tab), O.volume_points(m, tab, np.arange(m.E)), rtol=1e-14, atol=1e-15)


def test_workspace_is_given_back(gpu_ctx):
    """The kept workspace counts as in use and makes room for an allocation
    that needs its bytes: at the smallest budget (in steps of 2 %) that a mesh
    can be built in, the same mesh can be built again after a load."""
    m = M.structured_box_mesh(n=12)
    tab = R.rule_tables(m.etype, 3)
    budget = 1 << 20
    while True:
        ctx = _lib.Context(hbm_budget=budget)
        try:
            dev = _lib.DeviceMesh(ctx, m.coords, m.etype, m.conn)
            break
        except _lib.LLFEMError as e:
            assert e.code == _lib.ENOMEM
            ctx.close()
            budget += budget // 50
    bare = ctx.bytes_in_use()
    f = dev.body(tab, g=[1.0, 0.0, 0.0])
    assert ctx.bytes_in_use() > bare
    dev.close()
    assert ctx.bytes_in_use() > 0.02 * budget          # what is kept would not fit beside a second build
    dev = _lib.DeviceMesh(ctx, m.coords, m.etype, m.conn)
    assert np.array_equal(dev.body(tab, g=[1.0, 0.0, 0.0]), f)
    dev.close()
    ctx.close()
