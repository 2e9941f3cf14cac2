"""FP64 products of the PCG engine's updates at the row lengths where their
lanes per row change (8 below 9 blocks a row on average, 16 below 20, else 32):
separate hexahedra (8 blocks a row) and wedges (6), rods of one and of two by
two hexahedra (11.8 and 16.0), tet4 (11.8), a plate of one layer of hexahedra
(17.4), a block of hexahedra (20.8), hex27 (49).  The reference is the host's FP64
residual of the assembled matrix; 1e-10 is asked for, so a product that misses
an entry of K would be reported as a residual it is not."""
import numpy as np
import pytest
import scipy.sparse as sp

from lowlevelfem import _lib
from lowlevelfem import mesh as M
from lowlevelfem import refelem as R

pytestmark = pytest.mark.gpu


def _separate(elem, count):
    b = M.structured_box_mesh(n=1, elem=elem)
    conn = np.asarray(b.conn)[0]
    nodes = np.unique(conn)
    x, c = np.asarray(b.coords)[nodes], np.searchsorted(nodes, conn)
    coords = np.concatenate([x + [2.0 * k, 0.0, 0.0] for k in range(count)])
    return coords, b.etype, np.stack([c + nodes.size * k for k in range(count)])


def _box(**kw):
    m = M.structured_box_mesh(**kw)
    return m.coords, m.etype, m.conn


CASES = [("hex8 separate", lambda: _separate("hex", 33), 8), ("wedge separate", lambda: _separate("prism", 50), 8),
         ("rod", lambda: _box(cells=(1, 1, 40)), 16), ("rod 2x2", lambda: _box(cells=(2, 2, 30)), 16),
         ("tet4", lambda: _box(n=6, elem="tet"), 16), ("plate", lambda: _box(cells=(40, 40, 1)), 16),
         ("block", lambda: _box(cells=(7, 7, 7)), 32), ("hex27", lambda: _box(n=4, order=2), 32)]


@pytest.mark.parametrize("method", [_lib.PCG_MIXED_RELIABLE, _lib.PCG_F32OP_RELIABLE])
@pytest.mark.parametrize("label,make,lanes", CASES, ids=[c[0] for c in CASES])
def test_update_products(gpu_ctx, label, make, lanes, method):
    coords, etype, conn = make()
    dev = _lib.DeviceMesh(gpu_ctx, coords, etype, conn)
    val, _ = dev.assemble(_lib.OP_STIFFNESS, R.rule_tables(etype, 5), E=1.0)
    cp, rv = dev.pattern()
    n = 3 * len(coords)
    row = val.size / 9 / len(coords)
    assert lanes == (32 if row >= 20 else 16 if row >= 9 else 8)
    K = sp.csc_matrix((val, rv, cp), shape=(n, n))
    rng = np.random.default_rng(len(coords))
    f = rng.uniform(-1.0, 1.0, n)
    # every second node held: three corners or more of each separate element
    fixed = (3 * np.arange(0, len(coords), 2)[:, None] + np.arange(3)).ravel()
    ufix = rng.uniform(-1e-3, 1e-3, fixed.size)
    u, st = dev.solve(f, fixed, ufix, method=method, reltol=1e-10)
    free = np.ones(n, bool)
    free[fixed] = False
    u0 = np.zeros(n)
    u0[fixed] = ufix
    b = (f - K @ u0)[free]
    r = np.linalg.norm((K @ u - f)[free])
    assert np.array_equal(u[fixed], ufix)
    assert r <= 2e-10 * np.linalg.norm(b)
    # the reported residual is of the same product; both sides round each term of a row's sum
    eps = 2 * np.diff(cp).max() * 2.0 ** -53 * np.linalg.norm((abs(K) @ abs(u) + abs(f))[free])
    assert abs(r - st.relres * np.linalg.norm(f[free])) <= eps
    dev.close()
