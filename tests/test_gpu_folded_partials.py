"""Solves with more partial sums than a kernel's blocks sum by themselves, where
a launch of its own folds them first.

FP64 solver: a block walks up to eight groups of 256 / lanes rows, so that 2,048
partials remain; above 16,384 groups a block takes one and the partials are
folded: 2^19 rows at 8 lanes, 2^18 at 16, 2^17 at 32.  Cases on both sides, with
partials that 64 folding blocks do not share evenly.  Engine: above 4,096 blocks
of 16 nodes; FP32 operator with FP64 vectors here.

The reference is the host's FP64 residual.  A fold that loses or repeats a
partial gives a wrong p.Kp: the recursion then no longer follows b - K x, and the
true residual stays orders above the recursive one."""
import numpy as np
import pytest
import scipy.sparse as sp

from lowlevelfem import _lib
from lowlevelfem import mesh as M
from lowlevelfem import refelem as R
from test_gpu_csc_rows import _matrix

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,half,lanes", [(524_288, 3, 8), (524_289, 3, 8), (600_007, 11, 8), (262_144, 27, 16),
                                          (262_161, 27, 16), (131_072, 66, 32), (131_081, 66, 32)])
def test_csc(gpu_ctx, n, half, lanes):
    K = _matrix(n, half)
    row = K.nnz / n
    assert lanes == (32 if row >= 128 else 16 if row >= 48 else 8)
    f = np.random.default_rng(1).uniform(-1.0, 1.0, n)
    fixed = np.arange(0, n, 1001)
    cp, rv = K.indptr.astype(np.int64), K.indices.astype(np.int64)
    u, st = _lib.solve_csc(gpu_ctx, cp, rv, K.data, f, fixed, reltol=1e-12)
    r = K @ u - f
    r[fixed] = 0.0
    assert np.linalg.norm(r) <= 2e-12 * np.linalg.norm(f)
    u2, st2 = _lib.solve_csc(gpu_ctx, cp, rv, K.data, f, fixed, reltol=1e-12)
    assert np.array_equal(u, u2) and st2.iterations == st.iterations


# hex8, 32 lanes: 125,000 nodes (15,625 groups) and 132,651 (16,582); engine 7,813 and 8,291 blocks; 68,921 nodes and
# 64,000: engine 4,308 and 4,000
@pytest.mark.parametrize("n,method", [(49, _lib.PCG_JACOBI_FP64), (50, _lib.PCG_JACOBI_FP64),
                                      (50, _lib.PCG_MIXED_REFINE), (39, _lib.PCG_F32OP_RELIABLE),
                                      (40, _lib.PCG_F32OP_RELIABLE), (50, _lib.PCG_F32OP_RELIABLE)])
def test_panels(gpu_ctx, n, method):
    m = M.structured_box_mesh(n=n)
    dev = _lib.DeviceMesh(gpu_ctx, m.coords, m.etype, m.conn)
    val, _ = dev.assemble(_lib.OP_STIFFNESS, R.rule_tables(m.etype, 3), E=1.0)
    cp, rv = dev.pattern()
    K = sp.csc_matrix((val, rv, cp), shape=(3 * m.N, 3 * m.N))
    f = np.random.default_rng(n).uniform(-1.0, 1.0, 3 * m.N)
    left = m.nodes_on("left")
    fixed = (3 * left[:, None] + np.arange(3)).ravel()
    u, st = dev.solve(f, fixed, method=method, reltol=1e-10)
    r = K @ u - f
    r[fixed] = 0.0
    f0 = f.copy()
    f0[fixed] = 0.0
    assert np.linalg.norm(r) <= 2e-10 * np.linalg.norm(f0)
    u2, st2 = dev.solve(f, fixed, method=method, reltol=1e-10)
    assert np.array_equal(u, u2) and st2.iterations == st.iterations
    dev.close()
