"""Mixed-precision PCG engine and V-cycle kernels at the sizes where their
launch shape changes: fewer nodes than a row block, remainders of 16 rows,
more than 4,096 row blocks (partials folded first).  The reference is the FP64
residual of the assembled matrix on the host; the solver is asked for 1e-10."""
import numpy as np
import pytest
import scipy.sparse as sp

from lowlevelfem import _lib
from lowlevelfem import mesh as M
from lowlevelfem import refelem as R

pytestmark = pytest.mark.gpu


# nodes: 8, 27, 64 (4 row blocks), 125 (13 rows left), 216 (all levels in the tail kernel), 343 and 729 (the fine one
# not), 64,000 (4,000 blocks, a level between), 68,921 (4,308)
@pytest.mark.parametrize("method", [_lib.PCG_MIXED_RELIABLE, _lib.PCG_AMG_RELIABLE])
@pytest.mark.parametrize("n", [1, 2, 3, 4, 5, 6, 8, 39, 40])
def test_row_blocks(gpu_ctx, n, method):
    m = M.structured_box_mesh(n=n)
    dev = _lib.DeviceMesh(gpu_ctx, m.coords, m.etype, m.conn)
    val, _ = dev.assemble(_lib.OP_STIFFNESS, R.rule_tables(m.etype, 3), E=1.0)
    cp, rv = dev.pattern()
    K = sp.csc_matrix((val, rv, cp), shape=(3 * m.N, 3 * m.N))
    f = np.random.default_rng(n).uniform(-1.0, 1.0, 3 * m.N)
    left = m.nodes_on("left")
    fixed = (3 * left[:, None] + np.arange(3)).ravel()
    ufix = np.linspace(-1e-3, 1e-3, fixed.size)
    u, st = dev.solve(f, fixed, ufix, method=method, reltol=1e-10)
    free = np.ones(3 * m.N, bool)
    free[fixed] = False
    u0 = np.zeros(3 * m.N)
    u0[fixed] = ufix
    b = (f - K @ u0)[free]
    assert np.array_equal(u[fixed], ufix)
    assert np.linalg.norm((K @ u - f)[free]) <= 2e-10 * np.linalg.norm(b)
    u2, st2 = dev.solve(f, fixed, ufix, method=method, reltol=1e-10)
    assert np.array_equal(u, u2) and st2.iterations == st.iterations
    dev.close()


# 28^3 x 6 tet10: 185,193 nodes, more than 131,072 aggregate pairs on the fine
# level (16 lanes a pair); 12^3: a wave a pair on every level.  A coarse
# operator that lacks a block or counts one twice is no Galerkin product: the
# cycle would then converge slowly or not at all, so the iterations of the
# larger box stay within twice those of the smaller.
def test_galerkin_lanes(gpu_ctx):
    its = []
    for n in (12, 28):
        m = M.structured_box_mesh(n=n, elem="tet", order=2)
        dev = _lib.DeviceMesh(gpu_ctx, m.coords, m.etype, m.conn)
        dev.assemble(_lib.OP_STIFFNESS, R.rule_tables(m.etype, 2), E=1.0, copy_out=False)
        f = np.random.default_rng(n).uniform(-1.0, 1.0, 3 * m.N)
        left = m.nodes_on("left")
        fixed = (3 * left[:, None] + np.arange(3)).ravel()
        _, st = dev.solve(f, fixed, method=_lib.PCG_AMG_RELIABLE, reltol=1e-10)
        assert st.relres <= 1e-10
        its.append(st.iterations)
        dev.close()
    assert its[1] <= 2 * its[0]
