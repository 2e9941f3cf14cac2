"""FP64 Jacobi-PCG kernels at the sizes where their launch shape changes:
lanes per row (8, 16, 32 by the average row), more partials than a block sums
by itself, and the smallest systems.  The reference is scipy's direct solve;
the tolerance follows from the residual: ||e|| / ||u|| <= cond(K_ff) * relres,
cond of these small boxes and banded matrices below 1e5, relres 1e-12."""
import numpy as np
import pytest
import scipy.sparse as sp
import scipy.sparse.linalg as spl

from lowlevelfem import _lib
from lowlevelfem import mesh as M
from lowlevelfem import refelem as R

pytestmark = pytest.mark.gpu


def _check(K, f, fixed, u, ufix):
    n = f.size
    free = np.ones(n, bool)
    free[fixed] = False
    ref = np.zeros(n)
    ref[fixed] = ufix
    b = (f - K @ ref)[free]
    ref[free] = spl.spsolve(K[free][:, free].tocsc(), b)
    assert np.array_equal(u[fixed], ref[fixed])
    assert np.linalg.norm(u - ref) <= 1e-7 * np.linalg.norm(ref)


def _banded(n, half, seed=0):
    """Symmetric, strictly diagonally dominant, 2 half + 1 entries a row."""
    rng = np.random.default_rng(seed)
    K = sp.lil_matrix((n, n))
    for k in range(1, min(half, n - 1) + 1):
        K.setdiag(rng.uniform(-1.0, 1.0, n - k), k)
    K = (K + K.T).tocsc()
    return (K + sp.diags(np.asarray(abs(K).sum(axis=1)).ravel() + 1.0)).tocsc()


# average row 3 -> 8 lanes, 17 -> 16, 61 -> 32; 70,000 rows of 16 lanes are 4,375 partials; 1 and 3 rows
@pytest.mark.parametrize("n,half", [(1, 0), (3, 1), (257, 1), (70_001, 8), (2_001, 8), (16_500, 30)])
def test_csc_lanes(gpu_ctx, n, half):
    K = _banded(n, half)
    f = np.random.default_rng(1).uniform(-1.0, 1.0, n)
    fixed = np.arange(0, n, 7) if n > 1 else np.zeros(0, np.int64)
    ufix = np.linspace(-1.0, 1.0, fixed.size)
    u, st = _lib.solve_csc(gpu_ctx, K.indptr.astype(np.int64), K.indices.astype(np.int64), K.data, f, fixed, ufix,
                           reltol=1e-12)
    assert st.relres <= 1e-11
    _check(K, f, fixed, u, ufix)


# rows of about 15 (tet4), 27 (hex8) and 64 (hex27) blocks; 26^3 hex8: 2,461 partials
@pytest.mark.parametrize("elem,order,n,method", [("tet", 1, 5, 0), ("hex", 1, 4, 0), ("hex", 1, 26, 0), ("hex", 2, 3, 0),
                                                 ("prism", 1, 4, 1), ("tet", 2, 4, 1)])
def test_panel_lanes(gpu_ctx, elem, order, n, method):
    m = M.structured_box_mesh(n=n, elem=elem, order=order)
    dev = _lib.DeviceMesh(gpu_ctx, m.coords, m.etype, m.conn)
    val, _ = dev.assemble(_lib.OP_STIFFNESS, R.rule_tables(m.etype, 2 * order + 1), E=1.0)
    cp, rv = dev.pattern()
    K = sp.csc_matrix((val, rv, cp), shape=(3 * m.N, 3 * m.N))
    f = np.random.default_rng(2).uniform(-1.0, 1.0, 3 * m.N)
    left = m.nodes_on("left")
    fixed = (3 * left[:, None] + np.arange(3)).ravel()
    u, st = dev.solve(f, fixed, method=method, reltol=1e-12 if method == 0 else 1e-10)
    assert st.relres <= 1e-9
    if n < 20:
        _check(K, f, fixed, u, np.zeros(fixed.size))
    else:
        r = (K @ u - f)
        r[fixed] = 0.0
        assert np.linalg.norm(r) <= 1e-10 * np.linalg.norm(f)
    u2, st2 = dev.solve(f, fixed, method=method, reltol=1e-12 if method == 0 else 1e-10)
    assert np.array_equal(u, u2) and st2.iterations == st.iterations


def test_maxiter_is_reported(gpu_ctx):
    K = _banded(500, 8)
    f = np.ones(500)
    for maxiter in (1, 3, 8, 9):
        with pytest.raises(_lib.LLFEMError, match="maxiter reached"):
            _lib.solve_csc(gpu_ctx, K.indptr.astype(np.int64), K.indices.astype(np.int64), K.data, f,
                           np.zeros(0, np.int64), reltol=1e-30, maxiter=maxiter)
