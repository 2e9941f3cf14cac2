"""CSC solves at the row lengths and row counts where the lanes per row change:
20, 48 and 128 entries a row on average, 2^16 and 2^18 rows, on both sides of
each line.  The reference is the host's FP64 residual of the caller's matrix; 1e-12
is asked for of a strictly diagonally dominant one, whose recursion converges in
a few ten iterations, so that its residual is the true one to rounding."""
import numpy as np
import pytest
import scipy.sparse as sp

from lowlevelfem import _lib

pytestmark = pytest.mark.gpu


def _matrix(n, half, seed=0):
    """Symmetric, 2 half + 1 entries a row (fewer at the ends): bands whose
    distances grow, so that rows reach far."""
    rng = np.random.default_rng(seed)
    offs = np.unique(np.round(np.geomspace(1, max(2, min(n - 1, 40 * half)), 3 * half)).astype(int))
    offs = np.sort(rng.choice(offs, half, replace=False))
    U = sp.diags([rng.uniform(-1.0, 1.0, n - k) for k in offs], offs, shape=(n, n), format="csr")
    K = (U + U.T).tocsr()
    return (K + sp.diags(np.asarray(abs(K).sum(axis=1)).ravel() * 1.2 + 0.1)).tocsc()


CASES = [(5_000, 9, 8), (5_000, 11, 16), (5_000, 23, 16), (5_000, 25, 32), (5_000, 66, 32),
         (65_536, 24, 32), (65_537, 24, 16), (70_000, 66, 32), (262_144, 12, 16), (262_145, 12, 8), (262_145, 9, 8)]


@pytest.mark.parametrize("n,half,lanes", CASES)
def test_residual(gpu_ctx, n, half, lanes):
    K = _matrix(n, half)
    row = K.nnz / n
    rule = 32 if row >= 128 else (32 if n <= 65_536 else 16) if row >= 48 else 16 if row >= 20 and n <= 262_144 else 8
    assert rule == lanes
    rng = np.random.default_rng(1)
    f = rng.uniform(-1.0, 1.0, n)
    fixed = np.arange(3, n, 101)
    ufix = rng.uniform(-1.0, 1.0, fixed.size)
    cp, rv = K.indptr.astype(np.int64), K.indices.astype(np.int64)
    u, st = _lib.solve_csc(gpu_ctx, cp, rv, K.data, f, fixed, ufix, reltol=1e-12)
    free = np.ones(n, bool)
    free[fixed] = False
    u0 = np.zeros(n)
    u0[fixed] = ufix
    assert np.array_equal(u[fixed], ufix)
    assert np.linalg.norm((K @ u - f)[free]) <= 2e-12 * np.linalg.norm((f - K @ u0)[free])
    u2, st2 = _lib.solve_csc(gpu_ctx, cp, rv, K.data, f, fixed, ufix, reltol=1e-12)
    assert np.array_equal(u, u2) and st2.iterations == st.iterations
